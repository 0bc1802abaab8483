// emu_solo.cpp -- runs the one-workgroup engine (engine_solo.hpp) under the CPU wave emulator.
// TEST INFRASTRUCTURE ONLY. Built by tests/emu/Makefile into tests/emu/libemu_solo.so.
#include "wave_emu.hpp"
#if !defined(__clang__)
template <class T, class V>
inline T __hip_atomic_fetch_or(T* p, V v, int, int) { return __atomic_fetch_or(p, (T)v, __ATOMIC_SEQ_CST); }
#endif
#include "engine_solo.hpp"

#include <vector>

using namespace rcm;

namespace {
template <class G>
int run(int32_t count, const int32_t* n, const int64_t* rp_off, const int64_t* ci_off, const int32_t* rpc,
        const int32_t* cic, const int32_t* start, int32_t workers, int32_t mode, int32_t speculate, int32_t* perm_cat,
        int32_t* info, double timeout_s) {
  int64_t tot = 0;
  for (int k = 0; k < count; ++k) tot += n[k];
  std::vector<int32_t> perm(tot, -1);
  std::vector<uint64_t> qinfo(tot, 0x5A5A5A5A5A5A5A5Aull);
  std::vector<Control> ctl(count);
  std::vector<JobDesc> jobs(count);
  std::vector<int32_t> list(count);
  int64_t po = 0;
  for (int k = 0; k < count; ++k) {
    if (n[k] > G::B) return -2;
    JobDesc& J = jobs[k];
    J = JobDesc{};
    J.row_ptr = rpc + rp_off[k];
    J.col_idx = cic + ci_off[k];
    for (int32_t i = 0; i < n[k]; ++i)
      if (J.row_ptr[i + 1] - J.row_ptr[i] > kSoloMaxRow) return -3;
    J.perm = perm.data() + po;
    J.qinfo = qinfo.data() + po;
    J.ctl = &ctl[k];
    J.n = n[k];
    po += n[k];
    list[k] = count - 1 - k;
  }
  uint32_t next = 7;
  SoloManyArgs m{};
  m.jobs = jobs.data();
  m.list = list.data();
  m.starts = start;
  m.next = &next;
  m.count = count;
  m.mode = mode;
  m.speculate = speculate;
  m.budget_ticks = (uint64_t)(timeout_s * 1e8);
  emu::launch(1, 64, false, k_solo_reset, &next);
  emu::emu_lds_bytes = sizeof(SoloSmem<G>);
  emu::launch((unsigned)workers, G::T, true, k_solo_many<G>, m);
  emu::emu_lds_bytes = 256 * 1024;
  std::memcpy(perm_cat, perm.data(), sizeof(int32_t) * tot);
  for (int k = 0; k < count; ++k) {
    const int32_t v[6] = {(int32_t)ctl[k].error,  (int32_t)ctl[k].placed, (int32_t)ctl[k].nbatches,
                          ctl[k].start, ctl[k].sweeps, ctl[k].passes};
    std::memcpy(info + 6 * k, v, sizeof(v));
  }
  return 0;
}
}  // namespace

extern "C" {
// Orders `count` concatenated matrices, one workgroup each. geo: 0 = the geometry of small chunks (128 threads, 256
// slots, a ring of 64 entries: chunks, their remainders and the ring's overflow at small sizes), 1 = the library's.
// perm_cat: matrix k's order at sum_{i<k} n[i]; info[6 k ..] = error, placed, steps, start, sweeps, passes.
int emu_run_solo(int32_t count, const int32_t* n, const int64_t* rp_off, const int64_t* ci_off, const int32_t* rpc,
                 const int32_t* cic, const int32_t* start, int32_t workers, int32_t mode, int32_t speculate,
                 int32_t geo, int32_t* perm_cat, int32_t* info, double timeout_s) {
  if (count <= 0 || workers <= 0) return -1;
  return geo ? run<SoloGeo<512, 2048, 1 << 16>>(count, n, rp_off, ci_off, rpc, cic, start, workers, mode, speculate,
                                               perm_cat, info, timeout_s)
             : run<SoloGeo<128, 256, 1 << 16, 64>>(count, n, rp_off, ci_off, rpc, cic, start, workers, mode,
                                                   speculate, perm_cat, info, timeout_s);
}
}
