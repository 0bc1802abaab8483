// emu_solo.cpp -- runs the one-workgroup engine (engine_solo.hpp) under the CPU wave emulator.
// TEST INFRASTRUCTURE ONLY. Built by tests/emu/Makefile into tests/emu/libemu_solo.so.
#include "wave_emu.hpp"
#if !defined(__clang__)
template <class T, class V>
inline T __hip_atomic_fetch_or(T* p, V v, int, int) { return __atomic_fetch_or(p, (T)v, __ATOMIC_SEQ_CST); }
#endif
#include <unistd.h>
// holds member emu_linger[1] (-1: all but the leader) up at place emu_linger[0], for a while, on levels of tag emu_linger[2]
// modulo 5
static int emu_linger[3] = {-1, -1, -1};
#define RCM_TEAM_LINGER(where, member, tag)                                                                      \
  do {                                                                                                           \
    if (emu_linger[0] == (where) && (emu_linger[1] < 0 ? (member) > 0 : emu_linger[1] == (member)) &&            \
        (int)((tag) % 5u) == emu_linger[2] && lane_id() == 0)                                                    \
      usleep(20000);                                                                                             \
    __builtin_amdgcn_s_waitcnt(0);                                                                               \
  } while (0)
#include "engine_team.hpp"

#include <vector>

using namespace rcm;

namespace {
template <class G>
int run(int32_t count, const int32_t* n, const int64_t* rp_off, const int64_t* ci_off, const int32_t* rpc,
        const int32_t* cic, const int32_t* start, int32_t workers, int32_t mode, int32_t speculate, SoloGiveUp give,
        int32_t* perm_cat, int32_t* info, double timeout_s) {
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
  m.give = give;
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

template <class G>
int team(int32_t n, const int32_t* rp, const int32_t* ci, int32_t start, int32_t workers, int32_t mode,
         int32_t speculate, int32_t wide, int32_t alone, int32_t cap, uint32_t tag0, int32_t* perm, int32_t* info,
         double timeout_s) {
  int32_t maxrow = 1;
  for (int32_t i = 0; i < n; ++i) maxrow = std::max(maxrow, rp[i + 1] - rp[i]);
  if (maxrow > kSoloMaxRow || workers > kTeamMax) return -3;
  std::vector<uint64_t> claim((size_t)n, 0x5A5A5A5A5A5A5A5Aull);
  const uint64_t old = tag0 ? (uint64_t)tag0 << 32 : 0x5A5A5A5A5A5A5A5Aull;
  std::vector<uint64_t> s0((size_t)kTeamMax * cap * 2, old), s1((size_t)kTeamMax * cap * 2, old),
      words((size_t)kTeamMax * kTeamWordStride, old), rec(4, 0x5A5A5A5A5A5A5A5Aull);
  Control ctl;
  TeamArgs a{};
  a.row_ptr = rp;
  a.col_idx = ci;
  a.perm = perm;
  a.claim = claim.data();
  a.stage[0] = s0.data();
  a.stage[1] = s1.data();
  a.words = words.data();
  a.rec = rec.data();
  a.ctl = &ctl;
  a.n = n;
  a.cap = cap;
  a.members = workers;
  a.mode = mode;
  a.start = start;
  a.speculate = speculate;
  a.wide = wide;
  a.alone = (uint32_t)alone;
  a.tag0 = tag0;
  a.budget_ticks = (uint64_t)(timeout_s * 1e8);
  emu::launch(2, 64, false, k_team_init, a);
  emu::emu_lds_bytes = sizeof(TeamSmem<G>);
  emu::launch((unsigned)workers, G::T, true, k_team<G>, a);
  emu::emu_lds_bytes = 256 * 1024;
  const int32_t v[6] = {(int32_t)ctl.error, (int32_t)ctl.placed, (int32_t)ctl.nbatches, ctl.start,
                        ctl.sweeps, ctl.passes};
  std::memcpy(info, v, sizeof(v));
  return 0;
}
}  // namespace

extern "C" {
// Orders `count` concatenated matrices, one workgroup each. geo: 0 = the geometry of small chunks (128 threads, 256
// slots, a ring of 64 entries: chunks, their remainders and the ring's overflow at small sizes), 1 = the library's.
// wide_level, spare: when a matrix is given up. perm_cat: matrix k's order at sum_{i<k} n[i]; info[6 k ..] = error, placed,
// steps, start, sweeps, passes.
int emu_run_solo(int32_t count, const int32_t* n, const int64_t* rp_off, const int64_t* ci_off, const int32_t* rpc,
                 const int32_t* cic, const int32_t* start, int32_t workers, int32_t mode, int32_t speculate,
                 int32_t geo, uint32_t wide_level, uint32_t spare, int32_t* perm_cat, int32_t* info, double timeout_s) {
  if (count <= 0 || workers <= 0) return -1;
  const SoloGiveUp give{wide_level, spare, spare};
  return geo ? run<SoloGeo<1024, 4096, kSoloMaxN>>(count, n, rp_off, ci_off, rpc, cic, start, workers, mode, speculate,
                                                 give, perm_cat, info, timeout_s)
             : run<SoloGeo<128, 256, 1 << 16, 64>>(count, n, rp_off, ci_off, rpc, cic, start, workers, mode,
                                                   speculate, give, perm_cat, info, timeout_s);
}

void emu_team_linger(int where, int member, int phase) {
  emu_linger[0] = where;
  emu_linger[1] = member;
  emu_linger[2] = phase;
}

// A clock that every look moves on by `step` ticks, from 0 (step 0: the time again). Returns what the one before came to.
uint64_t emu_clock(uint64_t step) {
  emu::clock_step = step;
  return emu::clock_ticks.exchange(0);
}

// Orders one matrix with a team of `workers` workgroups (engine_team.hpp). wide: parents per member wanted, as a power of
// two. alone: slots of a level its leader takes on its own. cap: entries of a stage region. tag0 0 starts from memory that
// holds anything. geo: 0 = workgroups of one wave (256 slots), 1 = of two waves (512 slots). info = error, placed, levels,
// start, sweeps, passes.
int emu_run_team(int32_t n, const int32_t* rp, const int32_t* ci, int32_t start, int32_t workers, int32_t mode,
                 int32_t speculate, int32_t wide, int32_t alone, int32_t cap, uint32_t tag0, int32_t geo, int32_t* perm,
                 int32_t* info, double timeout_s) {
  return geo ? team<TeamGeo<128, 512>>(n, rp, ci, start, workers, mode, speculate, wide, alone, cap, tag0, perm, info,
                                       timeout_s)
             : team<TeamGeo<64, 256>>(n, rp, ci, start, workers, mode, speculate, wide, alone, cap, tag0, perm, info,
                                      timeout_s);
}
}
