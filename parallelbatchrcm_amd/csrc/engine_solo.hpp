// engine_solo.hpp -- one workgroup orders one whole matrix (device code): the engine of matrices of at most
// kSoloMaxN rows whose rows hold at most kSoloMaxRow entries.
//
// The batch engine (engine.hpp) spreads one matrix over many workgroups, so every BFS level pays several
// device-scope round trips between them (0.6 us from a store on one XCD to a load on another, 0.28 us for an atomic)
// and waits for its records and look-backs: 5-10 us a level, whatever the level's width. Here nothing leaves the
// workgroup: a level of up to S entries is one step of two dependent memory round trips (the parents' columns, the
// children's row bounds: 0.1 us each from this XCD's L2, 0.2-0.4 us from further) and four workgroup barriers
// (0.03 us each). Many matrices run side by side, one per workgroup.
//
//   Queue. perm is the BFS queue, as in engine.hpp. A step takes a chunk of it: the next parents of the current
//   level, at most T of them with at most S entries (slots) together. Slots are numbered in (parent, row entry)
//   order, which is the serial algorithm's (src/rcm_cpu.cpp:83-92). Each queue entry carries its row's begin and the
//   exclusive degree prefix over the queue, so slot offsets need no scan. The entries of the queue that are still to
//   be expanded stay in an LDS ring; when more than R wait, the new ones go to memory (qinfo) until they are used up.
//   Claims. A bitmap in LDS holds the visited nodes. The unvisited columns of a chunk meet in an LDS hash table whose
//   words hold the smallest slot claiming each child: chunks run one after another in queue order, so the smallest
//   slot of the chunk is the serial owner. No claim word lives in memory and no atomic leaves the CU.
//   Order. The owned children are packed in slot order, so siblings are neighbours (one child per parent on average);
//   each counts the earlier ones of larger and the later ones of smaller degree, which gives its place in the stable
//   valence sort (src/rcm_cpu.cpp:94-96).
//   Wide levels. Above 24,576 slots or so a level is work for the whole GPU, and a matrix with enough left is given up
//   (SoloGiveUp).
//   Start search. The sweeps of SimplePeripheral::findPeripheral (src/simple_peripheral.cpp:44-141) and the order run
//   in the same launch: the rule on the last 32 discovered nodes needs only the queue and the level boundaries.
#pragma once
#include "engine_many.hpp"

namespace rcm {

// Longest row: a child compares its degree with its siblings', so the work of a row grows with its square.
constexpr int32_t kSoloMaxRow = 64;
constexpr int kSoloDegBits = 7;  // bits of a degree up to kSoloMaxRow
constexpr int32_t kSoloMaxN = 1 << 18;  // the largest bitmap compiled (32 KB of LDS)

// T threads, S slots per chunk, bitmap of B nodes, R ring entries (power of two).
template <int T_, int S_, int B_, int R_ = 2048>
struct SoloGeo {
  static constexpr int T = T_, S = S_, B = B_, R = R_;
  static constexpr int W = T / kWave;
  static constexpr int EPT = S / T;
  static constexpr int NC = S / kWave;
  static constexpr int HB = __builtin_ctz((unsigned)S_);  // S hash words: a chunk has at most S distinct children
  static_assert(S % T == 0 && NC <= kWave && (S & (S - 1)) == 0 && (R & (R - 1)) == 0 && B % 32 == 0, "geometry");
  static_assert((1 << kSoloDegBits) > kSoloMaxRow, "degrees fit their field");
  static_assert(S >= kSoloMaxRow && S <= 65536, "any one parent fits a chunk");
};

// Which passes of a search the watchdog counts. In a symmetric matrix every sweep is longer than the one before or confirms
// it; in others the sweeps may repeat for ever, so one that does neither moves the deadline no further.
struct SearchPasses {
  uint32_t count, longest;  // 1 and 0 at first
  __device__ __forceinline__ void sweep(uint32_t lev, bool attempt) {  // the sweep after it is due, and an attempt's repeat
    if (lev <= longest) return;
    longest = lev;
    count += attempt ? 2u : 1u;
  }
};

// The watchdog of a workgroup, kept by thread 0. Its budget is for one pass over each matrix, as where every sweep is a
// launch of its own: a pass is to end within one budget, and the pass numbered p (from 1) of any matrix within p budgets of
// the launch.
struct SoloClock {
  uint64_t t0, budget, deadline;
  uint32_t* beat;      // pinned, or null: changes as passes begin, so that the host does not give a long search up
  uint32_t most;       // the largest p yet
  SearchPasses due;
  __device__ __forceinline__ void begin(uint64_t ticks, uint32_t* b) {
    t0 = wall_ticks();
    budget = ticks;
    deadline = t0 + ticks;
    beat = b;
    most = 1u;
  }
  __device__ __forceinline__ bool pass() {  // before one: whether it is too late for it
    most = max(most, due.count);
    const uint64_t now = wall_ticks(), end = t0 + budget * most;
    deadline = min(end, now + budget);
    return now > end;
  }
};

template <class G>
struct SoloSmem {
  uint32_t tab[G::S];            // hash: the smallest slot claiming a child, kNoSlot when free
  uint32_t sc[G::S];             // per slot: the child while the chunk claims; then the owned children, packed
  uint32_t ckey[G::S + 2];       // packed children: parent << kSoloDegBits | degree; child o at o + 1, ~0 around them
  uint32_t crb[G::S];            // packed children: row begin
  uint32_t cdx[G::S];            // packed children: degree prefix over the packed order
  uint64_t ring[G::R];           // per waiting queue entry: row begin | degree prefix << 32
  uint32_t vis[G::B / 32];       // visited nodes
  uint32_t pd[G::T];             // per parent of the chunk: row begin - first slot
  alignas(16) uint16_t mark[G::S];  // 1 + parent at its first slot, 0 elsewhere
  uint16_t cpar[G::NC];          // per 64 slots: 1 + the parent of the first of them
  uint64_t cinfo[G::NC];         // per 64 slots: owned children | their degree sum << 32
  int32_t levstart[64];          // first queue position of the last 64 levels
  uint32_t np, E, quit;          // of the chunk: parents, slots; the watchdog fired in the pass
  uint32_t late;                 // it fired between two passes
  SoloClock clk;
  int32_t job, cur;
};
constexpr uint32_t kNoSlot = ~0u;

// What a launch does with each matrix.
enum : int32_t { SOLO_RUN = 0, SOLO_SEARCH = 1, SOLO_ORDER = 2 };

struct SoloJob {
  const int32_t* row_ptr;
  const int32_t* col_idx;
  int32_t* perm;
  uint64_t* qinfo;  // overflow of the ring
  int32_t n;
};

struct RowBounds {
  int32_t b, e;
} __attribute__((packed, aligned(4)));

// The place of packed child o of cnt, key ckey[o + 1], among its siblings: earlier ones of larger degree go behind it,
// later ones of smaller degree before it. pos and dp (its place and degree prefix in packed order) are corrected. The
// nearest kSib on either side are read together; few parents have more children.
template <class K>
__device__ __forceinline__ void packed_place(const K& ckey, uint32_t o, uint32_t cnt, uint32_t key, uint32_t& pos,
                                             uint32_t& dp) {
  constexpr int kSib = 3;
  constexpr uint32_t dm = (1u << kSoloDegBits) - 1u;
  uint32_t f[kSib], h[kSib];
#pragma unroll
  for (int u = 0; u < kSib; ++u) {
    f[u] = ckey[o >= (uint32_t)u ? o - (uint32_t)u : 0u];
    h[u] = ckey[min(o + 2u + (uint32_t)u, cnt + 1u)];
  }
#pragma unroll
  for (int u = 0; u < kSib; ++u) {  // siblings are neighbours: beyond the last one the keys differ above dm
    if ((f[u] ^ key) <= dm && f[u] > key) {
      --pos;
      dp -= f[u] & dm;
    }
    if ((h[u] ^ key) <= dm && h[u] < key) {
      ++pos;
      dp += h[u] & dm;
    }
  }
  if ((f[kSib - 1] ^ key) <= dm)
    for (uint32_t u = o - (uint32_t)kSib;; --u) {
      const uint32_t x = ckey[u];
      if ((x ^ key) > dm) break;
      if (x > key) {
        --pos;
        dp -= x & dm;
      }
    }
  if ((h[kSib - 1] ^ key) <= dm)
    for (uint32_t u = o + 2u + (uint32_t)kSib;; ++u) {
      const uint32_t x = ckey[u];
      if ((x ^ key) > dm) break;
      if (x < key) {
        ++pos;
        dp += x & dm;
      }
    }
}

// Claims in the table: a child's word holds the smallest of its slots. hash_try offers slot j the word h and returns what
// held it; hash_settle goes on from there and returns the child's word. (A slot's sm.sc is stored before; slots of the
// same child meet at one word, so the search ends: S words, at most S children.)
template <class SM>
__device__ __forceinline__ uint32_t hash_try(SM& sm, uint32_t h, uint32_t j) {
  uint32_t old = kNoSlot;
  (void)__hip_atomic_compare_exchange_strong(&sm.tab[h], &old, j, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP);
  return old;
}
template <class G, class SM>
__device__ __forceinline__ uint32_t hash_settle(SM& sm, uint32_t h, uint32_t old, uint32_t child, uint32_t j) {
  while (old != kNoSlot) {
    if (sm.sc[old] == child) {  // taken by this child
      (void)__hip_atomic_fetch_min(&sm.tab[h], j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      break;
    }
    h = (h + 1) & (uint32_t)(G::S - 1);
    old = hash_try(sm, h, j);
  }
  return h;
}

// The queue and the chunk of one pass, the same in every thread.
struct SoloState {
  int32_t head, tail;      // queue positions [head, tail) wait
  int32_t lev, lev_end;    // level of the entry at head, and where that level ends
  uint32_t hdp, tdp;       // degree prefixes at head and tail
  int32_t ov_lo, ov_hi;    // queue positions [ov_lo, ov_hi) wait in qinfo, the others in the ring
  uint32_t np, E;          // the chunk: parents, slots
};

// Marks parent i (row begin rb) of the chunk as the owner of slots [so, se).
template <class G>
__device__ __forceinline__ void solo_mark(SoloSmem<G>& sm, uint32_t i, uint32_t rb, uint32_t so, uint32_t se) {
  sm.pd[i] = rb - so;
  if (se > so) {
    sm.mark[so] = (uint16_t)(i + 1);
    const uint32_t c = (so + kWave - 1) / kWave;  // a row of at most kSoloMaxRow slots holds one chunk start at most
    if (c * kWave < se) sm.cpar[c] = (uint16_t)(i + 1);
  }
}

// Takes the next chunk off the queue: parents from head on, within their level. Ends before a barrier.
template <class G>
__device__ __forceinline__ void solo_take(const SoloJob& J, SoloSmem<G>& sm, const SoloState& q) {
  constexpr int T = G::T, S = G::S, R = G::R;
  const int tid = threadIdx.x;
  const int32_t avail = min(q.lev_end - q.head, (int32_t)T);
  if (tid < avail) {
    const int32_t p = q.head + tid, p1 = p + 1;
    uint64_t e = sm.ring[p & (R - 1)];
    uint32_t dpn = (uint32_t)(sm.ring[p1 & (R - 1)] >> 32);
    if (q.ov_hi > q.head) {  // some wait in memory
      if (p >= q.ov_lo && p < q.ov_hi) e = ld_sync(&J.qinfo[p]);
      if (p1 >= q.ov_lo && p1 < q.ov_hi) dpn = (uint32_t)(ld_sync(&J.qinfo[p1]) >> 32);
    }
    if (p1 == q.tail) dpn = q.tdp;
    const uint32_t so = (uint32_t)(e >> 32) - q.hdp, se = dpn - q.hdp;
    if (se <= (uint32_t)S) {
      solo_mark<G>(sm, (uint32_t)tid, (uint32_t)e, so, se);
      if (tid + 1 == avail) {
        sm.np = (uint32_t)avail;
        sm.E = se;
      }
    } else if (so <= (uint32_t)S) {  // the first parent that does not fit
      sm.np = (uint32_t)tid;
      sm.E = so;
    }
  }
}

// Expands the marked chunk (at most KN * T slots): places its children and marks them as the next chunk when they are
// a whole level that fits one; otherwise they wait in the ring, or in qinfo when it is full. Returns whether the next
// chunk is marked. Starts and ends with every thread past a barrier.
template <class G, int KN>
__device__ __forceinline__ bool solo_step(const SoloJob& J, SoloSmem<G>& sm, SoloState& q, bool bfs) {
  constexpr int T = G::T, S = G::S, W = G::W, R = G::R;
  const int tid = threadIdx.x, ln = lane_id();
  const int wv = (int)wave_uniform((uint32_t)wave_id());
  const uint32_t nch = (q.E + kWave - 1) / kWave;
  const bool active = (uint32_t)wv < nch;
  // Slot j = 64 c + lane of 64-slot group c = kW + wave belongs to the parent of the prefix maximum of the marks. Its
  // column, then the claims: unvisited children into the hash table, smallest slot first, while their row bounds are
  // on the way.
  uint32_t cc[KN], par[KN], hp[KN], rb[KN], deg[KN];
  bool own[KN];
  if (active) {
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      const uint32_t c = (uint32_t)(k * W + wv), j = c * kWave + (uint32_t)ln;
      const uint32_t m = sm.mark[j], f = sm.cpar[c];
      par[k] = ln == 0 && c < nch ? max(m, f) : m;
      own[k] = j < q.E;
      if (m) sm.mark[j] = 0;
    }
#pragma unroll
    for (int k = 0; k < KN; ++k) par[k] = wave_incl_max(par[k]) - 1u;
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      cc[k] = 0;
      if (own[k]) cc[k] = (uint32_t)J.col_idx[sm.pd[par[k]] + (uint32_t)((k * W + wv) * kWave + ln)];
    }
#pragma unroll
    for (int k = 0; k < KN; ++k) hp[k] = sm.vis[cc[k] >> 5];
    RowBounds bd[KN];
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      own[k] = own[k] && !((hp[k] >> (cc[k] & 31u)) & 1u);
      hp[k] = (cc[k] * 2654435769u) >> (32 - G::HB);
      bd[k] = RowBounds{0, 0};
      if (own[k]) {
        sm.sc[(k * W + wv) * kWave + ln] = cc[k];
        bd[k] = *reinterpret_cast<const RowBounds*>(J.row_ptr + cc[k]);
      }
    }
    __asm__ volatile("" ::: "memory");  // a slot's child is in LDS before the slot can be found in the table
    uint32_t old[KN];
#pragma unroll
    for (int k = 0; k < KN; ++k) old[k] = own[k] ? hash_try(sm, hp[k], (uint32_t)((k * W + wv) * kWave + ln)) : kNoSlot;
#pragma unroll
    for (int k = 0; k < KN; ++k)
      hp[k] = hash_settle<G>(sm, hp[k], old[k], cc[k], (uint32_t)((k * W + wv) * kWave + ln));
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      rb[k] = (uint32_t)bd[k].b;
      deg[k] = (uint32_t)(bd[k].e - bd[k].b);
    }
  }
  __syncthreads();
  // owners: the slot its child's word holds. It frees the word (another slot of the same child finds neither its own
  // slot there nor in the freed word) and marks the child visited.
  uint64_t obal[KN];
  uint32_t dexc[KN];
  if (active) {
    uint32_t tw[KN];
#pragma unroll
    for (int k = 0; k < KN; ++k) tw[k] = sm.tab[hp[k]];
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      own[k] = own[k] && tw[k] == (uint32_t)((k * W + wv) * kWave + ln);
      if (own[k]) {
        sm.tab[hp[k]] = kNoSlot;
        (void)__hip_atomic_fetch_or(&sm.vis[cc[k] >> 5], 1u << (cc[k] & 31u), __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      obal[k] = ballot(own[k]);
    }
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      const uint32_t c = (uint32_t)(k * W + wv), d = own[k] ? deg[k] : 0u;
      const uint32_t inc = wave_incl_scan(d);
      dexc[k] = inc - d;
      if (ln == kWave - 1 && c < nch) sm.cinfo[c] = ((uint64_t)inc << 32) | (uint64_t)__popcll(obal[k]);
    }
  }
  __syncthreads();
  // the owned children in slot order, packed
  const uint64_t ci = (uint32_t)ln < nch ? sm.cinfo[ln] : 0ull;
  const uint32_t vc = (uint32_t)ci, vd = (uint32_t)(ci >> 32);
  const uint32_t ic = wave_incl_scan(vc), id = wave_incl_scan(vd);
  const uint32_t cnt = lane63(ic), dsum = lane63(id);
  if (active) {
    const uint32_t xc = ic - vc, xd = id - vd;
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      const uint32_t c = (uint32_t)(k * W + wv);
      const uint32_t pb = (uint32_t)__builtin_amdgcn_readlane((int)xc, (int)c);
      const uint32_t db = (uint32_t)__builtin_amdgcn_readlane((int)xd, (int)c);
      if (own[k]) {
        const uint32_t o = pb + (uint32_t)__popcll(obal[k] & lanemask_lt());
        sm.sc[o] = cc[k];
        sm.crb[o] = rb[k];
        sm.cdx[o] = db + dexc[k];
        sm.ckey[o + 1] = (par[k] << kSoloDegBits) | deg[k];
      }
    }
  }
  if (tid == 0) sm.ckey[cnt + 1] = ~0u;  // ends the last parent's siblings (ckey[0] starts the first one's)
  __syncthreads();
  // places: child o moves past the siblings around it that order the other way by degree
  const int32_t nhead = q.head + (int32_t)q.np, ntail = q.tail + (int32_t)cnt;
  const bool whole = q.head + (int32_t)q.np == q.lev_end && q.tail == q.lev_end;  // the level was this one chunk
  const bool direct = whole && cnt <= (uint32_t)T && dsum <= (uint32_t)S;
  const bool spill = !direct && (q.ov_hi > nhead || ntail - nhead > R);
  for (uint32_t o = (uint32_t)tid; o < cnt; o += T) {
    uint32_t pos = o, dp = sm.cdx[o];
    const uint32_t rbo = sm.crb[o], child = sm.sc[o], key = sm.ckey[o + 1];
    constexpr uint32_t dm = (1u << kSoloDegBits) - 1u;
    if (!bfs) packed_place(sm.ckey, o, cnt, key, pos, dp);
    const int32_t p = q.tail + (int32_t)pos;
    J.perm[p] = (int32_t)child;
    if (direct) {
      solo_mark<G>(sm, pos, rbo, dp, dp + (key & dm));
    } else {
      const uint64_t e = (uint64_t)rbo | ((uint64_t)(q.tdp + dp) << 32);
      if (spill)
        st_sync(&J.qinfo[p], e);
      else
        sm.ring[p & (R - 1)] = e;
    }
  }
  if (spill) {
    __builtin_amdgcn_s_waitcnt(0);
    if (q.ov_hi <= nhead) q.ov_lo = q.tail;
    q.ov_hi = ntail;
  }
  q.head = nhead;
  q.hdp += q.E;
  q.tail = ntail;
  q.tdp += dsum;
  if (direct) {  // the whole next level is the next chunk
    q.np = cnt;
    q.E = dsum;
  }
  __syncthreads();
  return direct;
}

// When a matrix is given up, for an engine of more workgroups: when more than `level` slots wait (about a level's; at least a
// chunk's) with more than `spare` entries of the matrix still to expand -- `growing`, if they are four times those expanded.
struct SoloGiveUp {
  uint32_t level, spare, growing;
};

// One pass over the matrix from `start`: the CM order (or the plain BFS order) into perm. Returns the nodes placed, or -1
// for a matrix given up; *levels the index of the last level. sm.quit is set when the watchdog fired.
template <class G>
__device__ __forceinline__ int32_t solo_pass(const SoloJob& J, SoloSmem<G>& sm, int32_t start, bool bfs, SoloGiveUp give,
                                             int32_t* levels, uint32_t* steps) {
  constexpr int T = G::T;
  const int tid = threadIdx.x;
  for (int32_t i = tid; i < (J.n + 31) / 32; i += T) sm.vis[i] = 0u;
  const uint32_t srb = (uint32_t)J.row_ptr[start], sdeg = (uint32_t)J.row_ptr[start + 1] - srb;
  __syncthreads();
  if (tid == 0) {
    sm.vis[start >> 5] |= 1u << (start & 31);
    sm.levstart[0] = 0;
    sm.quit = 0;
    sm.ckey[0] = ~0u;
    J.perm[0] = start;
    solo_mark<G>(sm, 0, srb, 0, sdeg);
  }
  __syncthreads();
  SoloState q{0, 1, 0, 1, 0, sdeg, 0, 0, 1, sdeg};
  bool marked = true;
  uint32_t step = 0;
  while (q.head < q.tail) {
    if (q.head == q.lev_end) {
      ++q.lev;
      q.lev_end = q.tail;
      if (tid == 0) sm.levstart[q.lev & 63] = q.head;
    }
    if (!marked) {
      const uint32_t waits = q.tdp - q.hdp;
      if (waits > give.level &&
          (uint32_t)J.row_ptr[J.n] - q.hdp > (waits / 4u > q.hdp ? give.growing : give.spare))
        return -1;
      solo_take<G>(J, sm, q);
      __syncthreads();
      q.np = wave_uniform(sm.np);
      q.E = wave_uniform(sm.E);
    }
    if ((++step & 63u) == 0u) {
      if (tid == 0) sm.quit = wall_ticks() > sm.clk.deadline ? 1u : 0u;
      __syncthreads();
      if (sm.quit) break;
    }
    marked = q.E <= (uint32_t)T ? solo_step<G, 1>(J, sm, q, bfs) : solo_step<G, G::EPT>(J, sm, q, bfs);
  }
  *levels = q.lev;
  *steps += step;
  return q.tail;
}

// One thread, as a pass after the first begins. The host allows 10 s beyond the budget; before 10 ms it need not know (the
// store to its memory takes 3 us, of a pass over a 100 x 100 grid's 290).
__device__ __forceinline__ void pass_beat(uint32_t* beat, uint64_t t0) {
  const uint64_t now = wall_ticks();
  if (beat && now - t0 > 1000000u) st_host(beat, (uint32_t)now);
}

// One matrix: the start search (SOLO_SEARCH), the order from `start` (SOLO_RUN), or both (SOLO_ORDER; `start` >= 0
// skips the search), or ERR_CAPACITY when it is given up. From sweep `speculate` on (0: never) a sweep of SOLO_ORDER is
// first run as a CM pass: when its eccentricity equals the previous sweep's it is the confirming sweep and the result. The
// results go to *ctl.
template <class G>
__device__ __forceinline__ void solo_matrix(const SoloJob& J, SoloSmem<G>& sm, int32_t mode, int32_t start,
                                            int32_t speculate, SoloGiveUp give, Control* ctl) {
  const int tid = threadIdx.x, ln = lane_id();
  for (int i = tid; i < G::S; i += G::T) sm.tab[i] = kNoSlot;
  for (int i = tid; i < G::S; i += G::T) sm.mark[i] = 0;
  // (the pass's first barrier orders these before their first use)
  const int32_t n = J.n;
  bool searching = mode != SOLO_RUN && start < 0 && n > 1, redo = false;
  int32_t cur = start >= 0 ? start : n > 1 ? n / 2 : 0;
  int32_t iters = start < 0 && n == 1 ? 1 : 0, passes = 0, placed = n, lev = 0;
  uint32_t steps = 0, lastdist = 0;
  bool expired = false;
  if (tid == 0) sm.clk.due = SearchPasses{1u, 0u};
  while (searching || mode != SOLO_SEARCH) {
    if (tid == 0) {  // a pass looks at the clock on every 64th step, and may have fewer
      sm.late = sm.clk.pass() ? 1u : 0u;
      if (passes > 0) pass_beat(sm.clk.beat, sm.clk.t0);
    }
    __syncthreads();
    expired = sm.late != 0;
    if (expired) break;
    if (searching && !redo) ++iters;
    const bool attempt = searching && !redo && mode == SOLO_ORDER && speculate > 0 && iters >= speculate;
    placed = solo_pass<G>(J, sm, cur, searching && !attempt, give, &lev, &steps);
    ++passes;
    expired = sm.quit != 0;
    if (placed != n || expired || !searching) break;
    if ((uint32_t)lev == lastdist) {  // cur is the start
      if (attempt || mode == SOLO_SEARCH) break;
      searching = false;
      if (tid == 0) ++sm.clk.due.count;
      continue;
    }
    if (tid == 0) sm.clk.due.sweep((uint32_t)lev, attempt);
    redo = attempt;  // a failed attempt is followed by the plain sweep from the same start
    if (redo) continue;
    lastdist = (uint32_t)lev;
    // the node of least row length among the last min(32, n - 1) of the last level, later ones winning ties
    __builtin_amdgcn_s_waitcnt(0);  // every wave's queue entries have reached the L2
    __syncthreads();
    if (wave_id() == 0) {
      const int32_t w = min(32, n - 1), p = n - w + ln;
      uint32_t key = ~0u;
      int32_t node = 0;
      if (ln < w && p >= sm.levstart[lev & 63]) {
        node = (int32_t)ld_sync(reinterpret_cast<const uint32_t*>(J.perm) + p);
        key = ((uint32_t)(J.row_ptr[node + 1] - J.row_ptr[node]) << 6) | (uint32_t)(63 - ln);
      }
      const uint32_t best = wave_min(key);
      if (key == best) sm.cur = node;
    }
    __syncthreads();
    cur = sm.cur;
  }
  if (tid == 0) {
    ctl->placed = (uint32_t)max(placed, 0);
    ctl->nbatches = steps ? steps : 1u;
    ctl->error = expired ? ERR_TIMEOUT : placed < 0 ? ERR_CAPACITY : ERR_NONE;
    ctl->start = cur;
    ctl->sweeps = iters;
    ctl->passes = passes;
    ctl->done = 1u;
    for (int i = 0; i < 9; ++i) ctl->diag[i] = 0u;
  }
  __syncthreads();
}

// One matrix in one launch.
template <class G>
__global__ __launch_bounds__(G::T) void k_solo(SoloJob J, int32_t mode, int32_t start, int32_t speculate,
                                               SoloGiveUp give, uint64_t budget_ticks, uint32_t* beat, Control* ctl) {
  using SM = SoloSmem<G>;
  RCM_LDS(SM, sm);
  if (threadIdx.x == 0) sm.clk.begin(budget_ticks, beat);
  solo_matrix<G>(J, sm, mode, start, speculate, give, ctl);
}

// Many matrices: workgroups take the jobs of the list in its order (largest first). A workgroup past the watchdog
// still takes the remaining jobs, each of which then ends at its first step with ERR_TIMEOUT, so every job of the
// list has a status.
struct SoloManyArgs {
  const JobDesc* jobs;
  const int32_t* list;    // the jobs of this launch
  const int32_t* starts;  // by job id
  uint32_t* next;         // position in the list, reset before the launch
  int32_t count;
  int32_t mode;
  int32_t speculate;
  SoloGiveUp give;
  uint64_t budget_ticks;
  uint32_t* beat;
};

__global__ void k_solo_reset(uint32_t* next) {
  if (threadIdx.x == 0) *next = 0u;
}

template <class G>
__global__ __launch_bounds__(G::T) void k_solo_many(SoloManyArgs m) {
  using SM = SoloSmem<G>;
  RCM_LDS(SM, sm);
  if (threadIdx.x == 0) sm.clk.begin(m.budget_ticks, m.beat);
  for (;;) {
    if (threadIdx.x == 0) {
      const uint32_t x = atomic_add_u32(m.next, 1u);
      sm.job = x < (uint32_t)m.count ? m.list[x] : -1;
    }
    __syncthreads();
    const int32_t j = (int32_t)wave_uniform((uint32_t)sm.job);
    if (j < 0) break;
    const JobDesc& D = m.jobs[j];
    const SoloJob J{D.row_ptr, D.col_idx, D.perm, D.qinfo, D.n};
    solo_matrix<G>(J, sm, m.mode, m.starts[j], m.speculate, m.give, D.ctl);  // ends with a barrier
  }
}

}  // namespace rcm
