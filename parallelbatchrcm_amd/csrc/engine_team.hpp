// engine_team.hpp -- a team of workgroups orders one matrix level by level (device code): the engine of larger
// matrices whose rows hold at most kSoloMaxRow entries.
//
// The batch engine (engine.hpp) lets the batches of a level overlap, at the price of about seven dependent
// device-scope round trips per level: tickets, records, claims, re-reads, look-backs (10 us a level on the 128^3
// stencil). A team instead expands a level in lockstep. Each member holds a contiguous part of the level's parents in
// LDS; the members claim, meet once (every claim of the level is made, and every member's parent count is known), and
// each orders the children it owns, which are its part of the next level. A meeting is one store and one poll of the
// members' words (1.35 us among 64 workgroups over all XCDs); what else a level waits for is the columns, the claim
// words twice and the row bounds.
//
//   Claims. claim[c] takes the minimum of (level, member, parent, row entry) over the entries that hold c. The parts
//   follow the queue in member order, so that is the order of the parents' queue positions, though the positions
//   themselves (the counts of the members before) are known only at the meeting; after it the entry whose code the
//   word holds owns c -- the serial rule (src/rcm_cpu.cpp:83-92). The codes of a later pass are below those of an
//   earlier one, so a pass needs no clearing.
//   Order. As in engine_solo.hpp: the owned children packed in slot order, siblings placed by (degree, slot).
//   Redistribution. When the level has outgrown its members or all levels before it, or left most members idle, or grown
//   lopsided, every member writes its children to its region of a double-buffered stage and their count to its word, and
//   the next level's parents are split evenly. Stage entries carry the tag of the level they are parents of, so a reader
//   that comes first polls the entry, and a writer publishes before it stores -- but for a part without children, whose
//   word may end the pass. A part that exceeds one chunk (T parents, S slots) also lives in the member's region, and is
//   expanded chunk by chunk.
//   Alone. Until the first redistribution of a pass its leader is the only member, and meets nobody: while the level is
//   narrow and the matrix has at most kTeamLocalN rows it claims in LDS, as engine_solo.hpp does (1.4 us a level against
//   3.2 through the claim words), and only stores the claims of what it places.
//   Membership. The workgroups that have started, in order of arrival; the first leads. Nobody waits for a workgroup
//   that has not started, so a launch ends whatever else runs on the GPU; the workgroups a level does without watch
//   the leader's word for the next redistribution.
// Measured on MI355X, whole calls, the batch engine before and a team after: one order of the 128^3 stencil 4.09 and 2.31 to
// 2.38 ms (379 levels), start search and order of a geometric graph of 1M points 23.0 and 14.2 to 14.8 ms, of a 48^3 stencil
// 3.4 and 1.9 ms.
#pragma once
#include "engine_solo.hpp"

// Where the tests hold a member up: between its word and its look at the others' (0 a meeting, 1 a redistribution),
// before a workgroup that joins reads the leader's record (2), and before a level's queue entries are stored (3).
// Nothing here relies on members keeping pace.
#ifndef RCM_TEAM_LINGER
#define RCM_TEAM_LINGER(where, member, tag)
#endif

namespace rcm {

constexpr int kTeamMax = 128;        // members: a lane polls the words of two neighbours
constexpr int kTeamPer = kTeamMax / kWave;
constexpr int kTeamWordStride = 16;  // a member's words lie on a 128-byte line of their own
constexpr int kTeamSplitWord = 2;    // behind the two of the meetings
constexpr int kTeamNodeBits = 24;    // of a node or count; with a degree or member count at most 32 bits
constexpr int kTeamPartBits = 18;    // of a parent's index in its member's part
constexpr int32_t kTeamLocalN = 1 << 18;  // the bitmap of the leader's local levels
constexpr int32_t kTeamMaxN = (1 << kTeamNodeBits) - 1;
constexpr int32_t kTeamMaxCap = 1 << kTeamPartBits;
static_assert(kSoloDegBits + kTeamNodeBits <= 32 && kTeamMax < 256, "fields of a stage entry and of a word");
static_assert(kTeamMax <= 1 << (32 - kTeamPartBits - kSoloDegBits), "fields of a claim code");

template <int T_, int S_>
struct TeamGeo {
  static constexpr int T = T_, S = S_;
  static constexpr int W = T / kWave;
  static constexpr int EPT = S / T;
  static constexpr int NC = S / kWave;
  static constexpr int HB = __builtin_ctz((unsigned)S_);
  static_assert((S & (S - 1)) == 0, "hash");
  static_assert(S % T == 0 && EPT >= 4 && NC <= kWave && S >= kSoloMaxRow && S <= 65536, "geometry");
};

struct TeamArgs {
  const int32_t* row_ptr;
  const int32_t* col_idx;
  int32_t* perm;
  uint64_t* claim;  // n words, all ~0 at the launch
  // parents of the levels of even and odd tags: kTeamMax regions of `cap` entries of two words, row begin | tag << 32 and
  // degree | node << 7 | tag << 32; no word holds a tag above tag0 at the launch (with tag0 0: anything)
  uint64_t* stage[2];
  // per member, zero at the launch. Words 0 and 1, levels of even and odd tags: tag << 32 | (the leader's: workgroups
  // started) << 24 | parents, its claims of that level made. A member may be through with the next level's claims before
  // another has read its word of this one, so they alternate; it is not through with the meeting after that, which needs
  // the other. Word 2: tag << 32 | next members << 24 | children, its part of a redistribution.
  uint64_t* words;
  uint64_t* rec;     // two records of two words: the state of a redistributed level for workgroups that join it
  Control* ctl;      // ticket, done and error zero at the launch
  int32_t n;
  int32_t cap;       // entries of a stage region
  int32_t members;   // at most this many
  int32_t mode, start, speculate;
  int32_t wide;      // parents per member wanted, as a power of two
  uint32_t alone;    // slots beyond which the leader shares its next local level
  uint32_t tag0;     // the first level's tag is tag0 + 1
  uint64_t budget_ticks;
  uint32_t* beat;    // as SoloClock's
};

template <class G>
struct TeamSmem {
  uint32_t sc[G::S];         // packed children: node
  uint32_t ckey[G::S + 2];   // packed children: parent << kSoloDegBits | degree; child o at o + 1, ~0 around them
  uint32_t crb[G::S];        // packed children: row begin
  uint32_t cdx[G::S];        // packed children: degree prefix over the packed order
  uint64_t pd[G::T];         // per parent of the chunk: row begin - first slot | first slot << 32
  uint32_t node[G::T];       // per parent of the chunk: the node
  alignas(16) uint16_t mark[G::S];  // 1 + parent at its first slot, 0 elsewhere
  uint16_t cpar[G::NC];      // per 64 slots: 1 + the parent of the first of them
  uint64_t cinfo[G::NC];     // per 64 slots: owned children | their degree sum << 32
  uint32_t tab[G::S];        // local levels: the smallest slot claiming a child, kNoSlot when free
  uint32_t vis[kTeamLocalN / 32];  // local levels: visited nodes
  uint32_t wtmp[G::W];
  uint32_t pre[kTeamMax + 1];  // redistribution: parents before each region
  uint32_t np, E;            // of a taken chunk: parents, slots
  uint32_t verdict, lost;
  uint64_t launch, t0, deadline;  // the watchdog
  SearchPasses due;          // thread 0 of the leader
  // of the meeting: parents of the members before, of all, of the largest part; workgroups started
  alignas(16) uint32_t met[4];
  uint32_t mnext, gnext;     // of a redistribution: parents of the next level, its members
  int32_t g, cur;
};

// One level, the same in every thread of a member.
struct TeamLevel {
  uint32_t tag;      // rises by one a level, over all passes
  int32_t members;   // that expand it
  int32_t pos;       // queue position of its first parent
  uint64_t base;     // of the level's claim codes
  bool bfs;
  // this member's part: `cnt` parents; marked: they are the chunk in LDS, of E slots; else they are entries
  // [p0, p0 + cnt) of `regions` stage regions from `region` on (sm.pre: parents before each)
  int32_t cnt, p0, regions, region;
  uint32_t E;
  bool marked;
  bool local;        // the leader, on its own since the pass began: sm.vis is up to date
};

enum : uint32_t { TEAM_ON = 0, TEAM_PASSED = 1, TEAM_STOP = 2 };

__device__ __forceinline__ uint64_t* team_word(const TeamArgs& a, int32_t g, int which) {
  return a.words + (size_t)g * kTeamWordStride + which;
}

__device__ __forceinline__ void team_fail(const TeamArgs& a, uint32_t err) {
  st_sync(&a.ctl->error, err);
  st_sync(&a.ctl->done, 1u);
}

// The watchdog (as SoloClock, in LDS: registers are short here): the leader says in ctl->passes how many passes are due; who
// runs out of time looks there.
template <class SM>
__device__ __forceinline__ bool team_late(const TeamArgs& a, SM& sm) {
  if (wall_ticks() <= sm.deadline) return false;
  const uint64_t due = (uint64_t)(uint32_t)ld_sync(&a.ctl->passes);
  sm.deadline = max(sm.deadline, sm.t0 + a.budget_ticks * due);
  return wall_ticks() > sm.deadline;
}

// One wave: whether to give up waiting (the launch is over, or the watchdog fires). Looked at on every 16th poll.
template <class SM>
__device__ __forceinline__ bool team_stop(const TeamArgs& a, SM& sm, uint32_t spin) {
  if (spin % 16u != 15u) return false;
  if (wave_uniform(ld_sync(&a.ctl->done))) return true;
  if (wave_uniform(team_late(a, sm) ? 1u : 0u)) {
    if (lane_id() == 0) team_fail(a, ERR_TIMEOUT);
    return true;
  }
  return false;
}

// Members to spread `width` parents over, of the `here` workgroups that have started.
__device__ __forceinline__ int32_t team_wanted(const TeamArgs& a, uint32_t width, uint32_t here) {
  const uint32_t w = (width + (1u << a.wide) - 1u) >> a.wide;
  return (int32_t)max(1u, min(w, min(here, (uint32_t)a.members)));
}

// Whether the children of a level of `width` parents, the largest part `most`, are redistributed: the members are too few
// for it, or a quarter of them would do, or one has twice its share, or it is many times all levels before: then
// its children may be as many times more, and most of them the first members', who claim first. (The limits are flat:
// growth from 1, 2 or 3 times the wanted part, imbalance of 2 or 3 above 2, 4 or 6 times it, 8 to 32 parents a part: within
// 10% of each other on 2D, 3D and geometric graphs, which outgrow what is behind them in their first levels only. Random
// graphs of 33k and 100k rows of 33 entries took 280 and 480 us an order without the last rule, 94 and 185 with it; by the
// batch engine 122 and 260.)
constexpr uint32_t kTeamGrowth = 4;
__device__ __forceinline__ bool team_split(const TeamArgs& a, const TeamLevel& lv, uint32_t width, uint32_t most,
                                           uint32_t here) {
  const int32_t want = team_wanted(a, width, here), members = lv.members;
  return (want > members && most > 2u << a.wide) || 4 * want <= members ||
         (most > 4u << a.wide && most * (uint32_t)members > 2u * width) ||
         (want > 1 && width > kTeamGrowth * (uint32_t)lv.pos);
}

// The words `which` of the first `members` members, two neighbours to a lane, until every tag is at least `tag`.
// TEAM_PASSED: one is above it.
struct TeamWords {
  uint64_t w[kTeamPer];
};
template <class SM>
__device__ __forceinline__ uint32_t team_poll(const TeamArgs& a, SM& sm, int which, uint32_t tag, int32_t members,
                                              TeamWords& r) {
  const int l0 = lane_id() * kTeamPer;
  for (uint32_t spin = 0;; ++spin) {
    bool early = false, late = false;
#pragma unroll
    for (int i = 0; i < kTeamPer; ++i) {
      r.w[i] = l0 + i < members ? ld_sync(team_word(a, l0 + i, which)) : (uint64_t)tag << 32;
      early = early || (uint32_t)(r.w[i] >> 32) < tag;
      late = late || (uint32_t)(r.w[i] >> 32) > tag;
    }
    if (ballot(late)) return TEAM_PASSED;
    if (!ballot(early)) return TEAM_ON;
    if (team_stop(a, sm, spin)) return TEAM_STOP;
  }
}
__device__ __forceinline__ uint32_t word_count(uint64_t w) { return (uint32_t)w & ((1u << kTeamNodeBits) - 1u); }

// The meeting: every member has made its claims of the level. False when the launch is over, or the pass (the words are
// those of a later one, sm.verdict is TEAM_PASSED): of a level without parents nobody waits for its members to read the
// words. Wave 0 has sm.met set when it passes the next barrier.
template <class G>
__device__ __forceinline__ bool team_meet(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, uint32_t here) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (lv.members == 1) {
    if (threadIdx.x == 0) {
      sm.met[0] = 0;
      sm.met[1] = sm.met[2] = (uint32_t)lv.cnt;
      sm.met[3] = here;
    }
    return true;
  }
  TeamWords r;
  if (wave_id() == 0) {
    if (lane_id() == 0)
      st_sync(team_word(a, sm.g, (int)(lv.tag & 1u)),
              ((uint64_t)lv.tag << 32) | (uint64_t)((here << kTeamNodeBits) | (uint32_t)lv.cnt));
    RCM_TEAM_LINGER(0, sm.g, lv.tag);
    const uint32_t v = team_poll(a, sm, (int)(lv.tag & 1u), lv.tag, lv.members, r);
    if (lane_id() == 0) sm.verdict = v;
  }
  __syncthreads();
  if (sm.verdict != TEAM_ON) return false;
  if (wave_id() == 0) {
    uint32_t c = 0, m = 0;
#pragma unroll
    for (int i = 0; i < kTeamPer; ++i) {
      c += word_count(r.w[i]);
      m = max(m, word_count(r.w[i]));
    }
    const uint32_t inc = wave_incl_scan(c), most = wave_max(m), tot = lane63(inc);
    const uint32_t hr = wave_uniform((uint32_t)r.w[0] >> kTeamNodeBits);
    uint32_t before = inc - c;
#pragma unroll
    for (int i = 0; i < kTeamPer; ++i) {
      if (lane_id() * kTeamPer + i == sm.g) sm.met[0] = before;
      before += word_count(r.w[i]);
    }
    if (lane_id() == 0) {
      sm.met[1] = tot;
      sm.met[2] = most;
      sm.met[3] = hr;
    }
  }
  return true;
}

// The children counts of a redistribution after the level `tag`, whose members are the first `members`: sm.pre, sm.mnext
// and the leader's sm.gnext. TEAM_PASSED when that is over for this workgroup (the others have gone on without it).
template <class G>
__device__ __forceinline__ uint32_t team_counts(const TeamArgs& a, TeamSmem<G>& sm, uint32_t tag, int32_t members) {
  if (wave_id() == 0) {
    TeamWords r;
    RCM_TEAM_LINGER(1, sm.g, tag);
    const uint32_t v = team_poll(a, sm, kTeamSplitWord, tag, members, r);
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < kTeamPer; ++i) c += word_count(r.w[i]);
    const uint32_t inc = wave_incl_scan(c);
    uint32_t before = inc - c;
#pragma unroll
    for (int i = 0; i < kTeamPer; ++i) {
      before += word_count(r.w[i]);
      if (lane_id() * kTeamPer + i < members) sm.pre[lane_id() * kTeamPer + i + 1] = before;
    }
    const uint32_t gn = wave_uniform(((uint32_t)r.w[0]) >> kTeamNodeBits), tot = lane63(inc);
    if (lane_id() == 0) {
      sm.pre[0] = 0;
      sm.verdict = v;
      sm.mnext = tot;
      sm.gnext = gn;
    }
  }
  __syncthreads();
  return sm.verdict;
}

// This member's even share of a redistributed level of `width` parents.
template <class G>
__device__ __forceinline__ void team_even(TeamSmem<G>& sm, TeamLevel& lv, int32_t width, int32_t members,
                                          int32_t regions) {
  const int32_t share = (int32_t)(((uint32_t)width + (uint32_t)members - 1u) / (uint32_t)members);
  lv.members = members;
  lv.p0 = min(width, sm.g * share);
  lv.cnt = min(width, lv.p0 + share) - lv.p0;
  lv.regions = regions;
  lv.region = 0;
  lv.marked = false;
}

// Marks parent i (row begin rb) of the chunk as the owner of slots [so, se).
template <class G>
__device__ __forceinline__ void team_mark(TeamSmem<G>& sm, uint32_t i, uint32_t rb, uint32_t so, uint32_t se,
                                          uint32_t node) {
  sm.pd[i] = (uint64_t)(rb - so) | ((uint64_t)so << 32);
  sm.node[i] = node;
  if (se > so) {
    sm.mark[so] = (uint16_t)(i + 1);
    const uint32_t c = (so + kWave - 1) / kWave;  // a row of at most kSoloMaxRow slots holds one chunk start at most
    if (c * kWave < se) sm.cpar[c] = (uint16_t)(i + 1);
  }
}

// Loads the parents from c0 on of the member's part from the stage, as far as their slots fit a chunk, and marks them;
// sm.np and sm.E tell how many parents and slots. Ends with a barrier. False when the launch is over.
template <class G>
__device__ __forceinline__ bool team_take(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, int32_t c0) {
  constexpr int T = G::T, S = G::S, W = G::W;
  const int tid = threadIdx.x;
  const int32_t avail = min(lv.cnt - c0, (int32_t)T);
  uint32_t d = 0, rb = 0, node = 0;
  if (tid < avail) {
    const int32_t p = lv.p0 + c0 + tid;
    int32_t lo = 0, hi = lv.regions;
    while (hi - lo > 1) {
      const int32_t mid = (lo + hi) >> 1;
      if ((int32_t)sm.pre[mid] <= p) lo = mid;
      else hi = mid;
    }
    const uint32_t first = lv.regions > 1 ? sm.pre[lo] : 0u;
    const uint64_t* e = a.stage[lv.tag & 1u] + 2 * ((size_t)(lv.region + lo) * (size_t)a.cap + (size_t)((uint32_t)p - first));
    uint64_t e0 = ld_sync(e), e1 = ld_sync(e + 1);
    for (uint32_t spin = 0; (uint32_t)(e0 >> 32) != lv.tag || (uint32_t)(e1 >> 32) != lv.tag; ++spin) {
      if (spin % 16u == 15u && (ld_sync(&a.ctl->done) || team_late(a, sm))) {
        sm.lost = 1;
        break;
      }
      e0 = ld_sync(e);
      e1 = ld_sync(e + 1);
    }
    rb = (uint32_t)e0;
    d = (uint32_t)e1 & ((1u << kSoloDegBits) - 1u);
    node = (uint32_t)e1 >> kSoloDegBits;
  }
  uint32_t se = wave_incl_scan(d);
  if (lane_id() == kWave - 1) sm.wtmp[wave_id()] = se;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < W; ++w) se += w < wave_id() ? sm.wtmp[w] : 0u;
  const uint32_t so = se - d;
  if (tid < avail) {
    if (se <= (uint32_t)S) {
      team_mark<G>(sm, (uint32_t)tid, rb, so, se, node);
      if (tid + 1 == avail) {
        sm.np = (uint32_t)avail;
        sm.E = se;
      }
    } else if (so <= (uint32_t)S) {  // the first parent that does not fit
      sm.np = (uint32_t)tid;
      sm.E = so;
    }
  }
  __syncthreads();
  if (sm.lost) {
    if (tid == 0 && !ld_sync(&a.ctl->done)) team_fail(a, ERR_TIMEOUT);
    return false;
  }
  return true;
}

// The slots of the marked chunk: slot j = 64 c + lane of 64-slot group c = kW + wave.
template <int KN>
struct TeamSlots {
  uint32_t cc[KN], par[KN], low[KN], rb[KN], deg[KN];  // low: the code's low word; of a local level, the hash word
  bool own[KN];
};

// Parents, columns and codes of the chunk whose first parent is c0 of the part.
template <class G, int KN>
__device__ __forceinline__ void team_expand(const TeamArgs& a, TeamSmem<G>& sm, int32_t c0, uint32_t E,
                                            TeamSlots<KN>& s) {
  constexpr int W = G::W;
  const int ln = lane_id();
  const int wv = (int)wave_uniform((uint32_t)wave_id());
  const uint32_t nch = (E + kWave - 1) / kWave;
  if ((uint32_t)wv >= nch) return;
  const uint32_t first = ((uint32_t)sm.g << kTeamPartBits) + (uint32_t)c0;
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    const uint32_t c = (uint32_t)(k * W + wv), j = c * kWave + (uint32_t)ln;
    const uint32_t m = sm.mark[j], f = sm.cpar[c];
    s.par[k] = ln == 0 && c < nch ? max(m, f) : m;
    s.own[k] = j < E;
    if (m) sm.mark[j] = 0;
  }
#pragma unroll
  for (int k = 0; k < KN; ++k) s.par[k] = wave_incl_max(s.par[k]) - 1u;
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    const uint32_t j = (uint32_t)((k * W + wv) * kWave + ln);
    s.cc[k] = s.low[k] = 0;
    if (s.own[k]) {
      const uint64_t pd = sm.pd[s.par[k]];
      s.cc[k] = (uint32_t)a.col_idx[(uint32_t)pd + j];
      s.low[k] = ((first + s.par[k]) << kSoloDegBits) | (j - (uint32_t)(pd >> 32));
    }
  }
}

// Claims: the word is read first; the atomic goes out only where it is still above the slot's code (codes only fall, so
// a stale word is an upper bound), with the child's row bounds in the same round trip. Sending every atomic at once, a
// round trip less, measured the same or slower: the GPU takes 27 random atomics a ns, but 250 loads.
template <class G, int KN>
__device__ __forceinline__ void team_claim(const TeamArgs& a, const TeamLevel& lv, uint32_t E, TeamSlots<KN>& s) {
  const int wv = (int)wave_uniform((uint32_t)wave_id());
  if ((uint32_t)wv * kWave >= E) return;
  uint64_t old[KN];
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    old[k] = 0;
    if (s.own[k]) old[k] = ld_sync(&a.claim[s.cc[k]]);
  }
  RowBounds b[KN];
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    const uint64_t code = lv.base | (uint64_t)s.low[k];
    s.own[k] = s.own[k] && old[k] > code;
    b[k] = RowBounds{0, 0};
    if (s.own[k]) {
      (void)atomic_min_u64(&a.claim[s.cc[k]], code);
      b[k] = *reinterpret_cast<const RowBounds*>(a.row_ptr + s.cc[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    s.rb[k] = (uint32_t)b[k].b;
    s.deg[k] = (uint32_t)(b[k].e - b[k].b);
  }
}

// Claims of a local level: unvisited children into the hash table, smallest slot first (engine_solo.hpp).
template <class G, int KN>
__device__ __forceinline__ void team_claim_local(const TeamArgs& a, TeamSmem<G>& sm, uint32_t E, TeamSlots<KN>& s) {
  constexpr int W = G::W;
  const int ln = lane_id();
  const int wv = (int)wave_uniform((uint32_t)wave_id());
  if ((uint32_t)wv * kWave >= E) return;
  uint32_t vw[KN];
#pragma unroll
  for (int k = 0; k < KN; ++k) vw[k] = sm.vis[s.cc[k] >> 5];
  RowBounds b[KN];
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    s.own[k] = s.own[k] && !((vw[k] >> (s.cc[k] & 31u)) & 1u);
    s.low[k] = (s.cc[k] * 2654435769u) >> (32 - G::HB);
    b[k] = RowBounds{0, 0};
    if (s.own[k]) {
      sm.sc[(k * W + wv) * kWave + ln] = s.cc[k];
      b[k] = *reinterpret_cast<const RowBounds*>(a.row_ptr + s.cc[k]);
    }
  }
  __asm__ volatile("" ::: "memory");  // a slot's child is in LDS before the slot can be found in the table
  uint32_t old[KN];
#pragma unroll
  for (int k = 0; k < KN; ++k)
    old[k] = s.own[k] ? hash_try(sm, s.low[k], (uint32_t)((k * W + wv) * kWave + ln)) : kNoSlot;
#pragma unroll
  for (int k = 0; k < KN; ++k)
    s.low[k] = hash_settle<G>(sm, s.low[k], old[k], s.cc[k], (uint32_t)((k * W + wv) * kWave + ln));
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    s.rb[k] = (uint32_t)b[k].b;
    s.deg[k] = (uint32_t)(b[k].e - b[k].b);
  }
}

// Wave 0: the member's word of the redistribution after this level, and the leader's record for those that join.
template <class G>
__device__ __forceinline__ void team_publish(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, uint32_t width,
                                             int32_t want, uint32_t children) {
  if (sm.g == 0) {
    if (lane_id() == 0) {
      uint64_t* r = a.rec + 2 * ((lv.tag + 1u) & 1u);
      st_sync(r, (uint64_t)((uint32_t)lv.pos + width) | ((uint64_t)(lv.bfs ? 1 : 0) << kTeamNodeBits) |
                     ((uint64_t)(uint32_t)lv.members << 32));
      st_sync(r + 1, lv.base + ((uint64_t)1 << 32));
    }
    __builtin_amdgcn_s_waitcnt(0);  // the record is there before the word says so
  }
  if (lane_id() == 0)
    st_sync(team_word(a, sm.g, kTeamSplitWord),
            ((uint64_t)lv.tag << 32) |
                (uint64_t)(((uint32_t)want << kTeamNodeBits) | children));
}

// What a member does with the children of its part.
struct TeamNext {
  uint32_t placed, E;  // children, their slots
  bool split;          // the next level is redistributed
  bool marked;         // they are the next chunk in LDS
};

// Places the children of the chunk (np parents from c0 of the part, every claim of the level is made) behind those placed
// already. only: the chunk is the whole part; last: its last one. LOCAL: of a local level. False when the member's region
// is full. Starts with every thread past a barrier, ends before one.
template <class G, int KN, bool LOCAL>
__device__ __forceinline__ bool team_place(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, int32_t c0,
                                           int32_t np, uint32_t E, TeamSlots<KN>& s, bool only, bool last,
                                           TeamNext& nx) {
  constexpr int T = G::T, S = G::S, W = G::W;
  const int tid = threadIdx.x, ln = lane_id();
  const int wv = (int)wave_uniform((uint32_t)wave_id());
  const uint32_t nch = (E + kWave - 1) / kWave;
  const bool active = (uint32_t)wv < nch;
  uint64_t obal[KN];
  uint32_t dexc[KN];
  if (active) {
    uint64_t now[KN];
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      now[k] = 0;
      if constexpr (LOCAL) now[k] = (uint64_t)sm.tab[s.low[k] & (uint32_t)(S - 1)];
      else if (s.own[k]) now[k] = ld_sync(&a.claim[s.cc[k]]);
    }
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      const uint32_t c = (uint32_t)(k * W + wv);
      if constexpr (LOCAL) {  // the owner frees its word and marks its child, here and for the levels to come
        s.own[k] = s.own[k] && (uint32_t)now[k] == c * kWave + (uint32_t)ln;
        if (s.own[k]) {
          sm.tab[s.low[k]] = kNoSlot;
          (void)__hip_atomic_fetch_or(&sm.vis[s.cc[k] >> 5], 1u << (s.cc[k] & 31u), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
          st_sync(&a.claim[s.cc[k]], lv.base);
        }
      } else {
        s.own[k] = s.own[k] && now[k] == (lv.base | (uint64_t)s.low[k]);
      }
      obal[k] = ballot(s.own[k]);
      const uint32_t d = s.own[k] ? s.deg[k] : 0u;
      const uint32_t inc = wave_incl_scan(d);
      dexc[k] = inc - d;
      if (ln == kWave - 1 && c < nch) sm.cinfo[c] = ((uint64_t)inc << 32) | (uint64_t)__popcll(obal[k]);
    }
  }
  __syncthreads();
  // the meeting's result is here too: the parents' queue positions, and where the children go
  const uint32_t before = sm.met[0], width = sm.met[1], most = sm.met[2], here = sm.met[3];
  if (here == 0) return false;  // the leader's watchdog fired
  const uint64_t ci = (uint32_t)ln < nch ? sm.cinfo[ln] : 0ull;
  const uint32_t vc = (uint32_t)ci, vd = (uint32_t)(ci >> 32);
  const uint32_t ic = wave_incl_scan(vc), id = wave_incl_scan(vd);
  const uint32_t cnt = lane63(ic), dsum = lane63(id);
  uint32_t share = width;
  if (LOCAL) {  // the leader knows the next level
    share = cnt;
    nx.split = dsum > a.alone && team_wanted(a, share, here) > 1;
    if (nx.split) {  // the claims stored are there before others read them
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
  } else {
    nx.split = team_split(a, lv, width, most, here);
  }
  const bool direct = only && !nx.split && cnt <= (uint32_t)T && dsum <= (uint32_t)S;
  if (!direct && nx.placed + cnt > (uint32_t)a.cap) {
    if (tid == 0) team_fail(a, ERR_CAPACITY);  // the others see it where they wait for this member
    return false;
  }
  const int32_t q0 = lv.pos + (int32_t)before + c0;
  if (q0 + np > a.n) {  // cannot happen: every node is owned once
    if (tid == 0) team_fail(a, ERR_CAPACITY);
    return false;
  }
  // Readers of a redistribution's children look at their tags, so its word goes out first. A part without children, though,
  // may be of the pass's last level: then the leader reads the queue as soon as it has the members' words, with no meeting
  // before, and the word waits for the part's queue entries (of all its chunks).
  const bool word = last && nx.split, barren = word && nx.placed + cnt == 0;
  const auto store_queue = [&]() {
    RCM_TEAM_LINGER(3, sm.g, lv.tag);
    if (tid < np) st_sync(&a.perm[q0 + tid], (int32_t)sm.node[tid]);
  };
  if (barren) {
    store_queue();
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (wv == 0 && word) team_publish<G>(a, sm, lv, width, team_wanted(a, share, here), nx.placed + cnt);
  if (!barren) store_queue();
  if (active) {
    const uint32_t xc = ic - vc, xd = id - vd;
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      const uint32_t c = (uint32_t)(k * W + wv);
      const uint32_t pb = (uint32_t)__builtin_amdgcn_readlane((int)xc, (int)c);
      const uint32_t db = (uint32_t)__builtin_amdgcn_readlane((int)xd, (int)c);
      if (s.own[k]) {
        const uint32_t o = pb + (uint32_t)__popcll(obal[k] & lanemask_lt());
        sm.sc[o] = s.cc[k];
        sm.crb[o] = s.rb[k];
        sm.cdx[o] = db + dexc[k];
        sm.ckey[o + 1] = (s.par[k] << kSoloDegBits) | s.deg[k];
      }
    }
  }
  if (tid == 0) sm.ckey[cnt + 1] = ~0u;  // ends the last parent's siblings (ckey[0] starts the first one's)
  __syncthreads();
  uint64_t* out = a.stage[(lv.tag + 1u) & 1u] + 2 * ((size_t)sm.g * (size_t)a.cap + nx.placed);
  const uint64_t tag = (uint64_t)(lv.tag + 1u) << 32;
  for (uint32_t o = (uint32_t)tid; o < cnt; o += T) {
    uint32_t pos = o, dp = sm.cdx[o];
    const uint32_t rbo = sm.crb[o], child = sm.sc[o], key = sm.ckey[o + 1];
    constexpr uint32_t dm = (1u << kSoloDegBits) - 1u;
    if (!lv.bfs) packed_place(sm.ckey, o, cnt, key, pos, dp);
    if (direct) {
      team_mark<G>(sm, pos, rbo, dp, dp + (key & dm), child);
    } else {
      st_sync(&out[2 * pos], tag | (uint64_t)rbo);
      st_sync(&out[2 * pos + 1], tag | (uint64_t)((child << kSoloDegBits) | (key & dm)));
    }
  }
  nx.placed += cnt;
  nx.E = dsum;
  nx.marked = direct;
  return true;
}

// The member's part of a level when it is one chunk, marked in LDS.
template <class G, int KN>
__device__ __forceinline__ bool team_chunk_local(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, uint32_t here,
                                                 TeamNext& nx) {
  TeamSlots<KN> s;
  team_expand<G, KN>(a, sm, 0, lv.E, s);
  team_claim_local<G, KN>(a, sm, lv.E, s);
  if (threadIdx.x == 0) {
    sm.met[0] = 0;
    sm.met[1] = sm.met[2] = (uint32_t)lv.cnt;
    sm.met[3] = here;
  }
  __syncthreads();
  return team_place<G, KN, true>(a, sm, lv, 0, lv.cnt, lv.E, s, true, true, nx);
}
template <class G, int KN>
__device__ __forceinline__ bool team_chunk(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, uint32_t here,
                                           TeamNext& nx) {
  TeamSlots<KN> s;
  team_expand<G, KN>(a, sm, 0, lv.E, s);
  team_claim<G, KN>(a, lv, lv.E, s);
  if (!team_meet<G>(a, sm, lv, here)) return false;
  return team_place<G, KN, false>(a, sm, lv, 0, lv.cnt, lv.E, s, true, true, nx);
}

// The part when it is more than one chunk: the claims of all of them, the meeting, then the children of each.
template <class G>
__device__ __forceinline__ bool team_chunks(const TeamArgs& a, TeamSmem<G>& sm, const TeamLevel& lv, int32_t np0,
                                            uint32_t E0, uint32_t here, TeamNext& nx) {
  constexpr int KN = G::EPT;
  TeamSlots<KN> s;
  int32_t np = np0;
  uint32_t e = E0;
  for (int32_t c0 = 0;;) {
    team_expand<G, KN>(a, sm, c0, e, s);
    team_claim<G, KN>(a, lv, e, s);
    c0 += np;
    if (c0 >= lv.cnt) break;
    __syncthreads();
    if (!team_take<G>(a, sm, lv, c0)) return false;
    np = (int32_t)sm.np;
    e = wave_uniform(sm.E);
  }
  if (!team_meet<G>(a, sm, lv, here)) return false;
  for (int32_t c0 = 0; c0 < lv.cnt;) {
    __syncthreads();
    if (!team_take<G>(a, sm, lv, c0)) return false;
    np = (int32_t)sm.np;
    e = wave_uniform(sm.E);
    team_expand<G, KN>(a, sm, c0, e, s);
    // row bounds again, for the slots that own their child
    if (wave_uniform((uint32_t)wave_id()) * kWave < e) {
#pragma unroll
      for (int k = 0; k < KN; ++k) {
        s.rb[k] = s.deg[k] = 0;
        s.own[k] = s.own[k] && ld_sync(&a.claim[s.cc[k]]) == (lv.base | (uint64_t)s.low[k]);
        if (s.own[k]) {
          const RowBounds b = *reinterpret_cast<const RowBounds*>(a.row_ptr + s.cc[k]);
          s.rb[k] = (uint32_t)b.b;
          s.deg[k] = (uint32_t)(b.e - b.b);
        }
      }
    }
    if (!team_place<G, KN, false>(a, sm, lv, c0, np, e, s, false, c0 + np >= lv.cnt, nx)) return false;
    c0 += np;
  }
  return true;
}

// One level as a member, and the state of the next one in lv. TEAM_PASSED: the pass is over (no parents in this level),
// or this workgroup is not a member of the next level. here: thread 0 of the leader, the workgroups started.
template <class G>
__device__ __forceinline__ uint32_t team_level(const TeamArgs& a, TeamSmem<G>& sm, TeamLevel& lv, uint32_t here) {
  TeamNext nx{0, 0, false, false};
  bool ok = true;
  if (lv.local && lv.cnt > 0 && !lv.marked) {  // too wide for one chunk: through the claim words from here on
    lv.local = false;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (lv.local) {
    ok = lv.E <= (uint32_t)G::T ? team_chunk_local<G, 1>(a, sm, lv, here, nx)
                                : team_chunk_local<G, G::EPT>(a, sm, lv, here, nx);
    if (!ok) return TEAM_STOP;
  } else if (lv.cnt > 0) {
    int32_t np = lv.cnt;
    if (!lv.marked) {
      if (!team_take<G>(a, sm, lv, 0)) return TEAM_STOP;
      np = (int32_t)sm.np;
      lv.E = wave_uniform(sm.E);
    }
    if (np < lv.cnt) ok = team_chunks<G>(a, sm, lv, np, lv.E, here, nx);
    else if (lv.E <= (uint32_t)G::T) ok = team_chunk<G, 1>(a, sm, lv, here, nx);
    else if (lv.E <= 2u * G::T) ok = team_chunk<G, 2>(a, sm, lv, here, nx);
    else ok = team_chunk<G, G::EPT>(a, sm, lv, here, nx);
    if (!ok) return TEAM_STOP;
  } else {
    if (!team_meet<G>(a, sm, lv, here)) return sm.verdict == TEAM_PASSED ? TEAM_PASSED : TEAM_STOP;
    __syncthreads();
    nx.split = team_split(a, lv, sm.met[1], sm.met[2], sm.met[3]);
    nx.marked = true;
    if (sm.met[3] == 0) return TEAM_STOP;
    if (wave_uniform((uint32_t)wave_id()) == 0u && nx.split)
      team_publish<G>(a, sm, lv, sm.met[1], team_wanted(a, sm.met[1], sm.met[3]), 0u);
  }
  const int32_t width = (int32_t)sm.met[1];
  __syncthreads();
  if (width == 0) return TEAM_PASSED;
  lv.pos += width;
  const uint32_t tag = lv.tag++;
  lv.base += 1ull << 32;
  if (nx.split) {
    const uint32_t v = team_counts<G>(a, sm, tag, lv.members);
    if (v != TEAM_ON) return v;
    const int32_t m = (int32_t)sm.mnext, gn = (int32_t)sm.gnext;
    if (m == 0 || gn <= sm.g) return TEAM_PASSED;
    team_even<G>(sm, lv, m, gn, lv.members);
    lv.local = false;
  } else {
    lv.cnt = (int32_t)nx.placed;
    lv.E = nx.E;
    lv.marked = nx.marked;
    lv.p0 = 0;
    lv.regions = 1;
    lv.region = sm.g;
    if (lv.members == 1 && lv.cnt == 0) return TEAM_PASSED;
  }
  return TEAM_ON;
}

// A workgroup that does not lead: watches the leader's word and takes part in the levels it is counted in.
template <class G>
__device__ __forceinline__ void team_help(const TeamArgs& a, TeamSmem<G>& sm) {
  uint32_t seen = a.tag0;
  for (;;) {
    if (wave_id() == 0) {
      uint32_t v = TEAM_ON, tag = 0, gn = 0;
      for (uint32_t spin = 0;; ++spin) {
        const uint64_t w = ld_sync(team_word(a, 0, kTeamSplitWord));
        tag = wave_uniform((uint32_t)(w >> 32));
        gn = wave_uniform((uint32_t)w >> kTeamNodeBits);
        if (tag > seen && (int32_t)gn > sm.g) break;
        if (team_stop(a, sm, spin)) {
          v = TEAM_STOP;
          break;
        }
        __builtin_amdgcn_s_sleep(4);
      }
      RCM_TEAM_LINGER(2, sm.g, tag);
      if (lane_id() == 0) {
        sm.verdict = v;
        sm.np = tag;
        sm.E = gn;
      }
    }
    __syncthreads();
    if (sm.verdict == TEAM_STOP) return;
    seen = sm.np;
    const int32_t gn = (int32_t)sm.E;
    const uint64_t r0 = ld_sync(a.rec + 2 * ((seen + 1u) & 1u)), r1 = ld_sync(a.rec + 2 * ((seen + 1u) & 1u) + 1);
    TeamLevel lv;
    lv.local = false;
    lv.tag = seen + 1u;
    lv.pos = (int32_t)((uint32_t)r0 & ((1u << kTeamNodeBits) - 1u));
    lv.bfs = ((r0 >> kTeamNodeBits) & 1u) != 0;
    lv.base = r1;
    const int32_t regions = (int32_t)wave_uniform((uint32_t)(r0 >> 32));
    __syncthreads();
    uint32_t v = team_counts<G>(a, sm, seen, regions);
    if (v == TEAM_ON) {
      const int32_t m = (int32_t)sm.mnext;
      if (m > 0) {
        team_even<G>(sm, lv, m, gn, regions);
        do {
          seen = lv.tag;
          v = team_level<G>(a, sm, lv, 0u);
        } while (v == TEAM_ON);
        // the leader's word of a redistribution after `seen` may count this workgroup again only later
      }
    }
    if (v == TEAM_STOP) return;
    __syncthreads();
  }
}

// The leader's pass from `start`: returns the nodes placed; *levels the index of the last level, *last its first queue
// position. *stop when the launch is over.
template <class G>
__device__ __forceinline__ int32_t team_pass(const TeamArgs& a, TeamSmem<G>& sm, int32_t start, bool bfs, uint32_t epoch,
                                             uint32_t* tag, int32_t* levels, int32_t* last, bool* stop) {
  const int tid = threadIdx.x;
  const uint32_t rb = (uint32_t)a.row_ptr[start], d = (uint32_t)a.row_ptr[start + 1] - rb;
  const uint64_t base = (uint64_t)epoch << 56;
  TeamLevel lv{++*tag, 1, 0, base + (1ull << 32), bfs, 1, 0, 1, 0, d, true, a.n <= kTeamLocalN};
  if (lv.local) {
    for (int32_t i = tid; i < (a.n + 31) / 32; i += G::T) sm.vis[i] = 0u;
    __syncthreads();
  }
  if (tid == 0) {
    if (lv.local) sm.vis[start >> 5] |= 1u << (start & 31);
    st_sync(&a.claim[start], base);
    team_mark<G>(sm, 0, rb, 0, d, (uint32_t)start);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int32_t lev = -1;
  uint32_t here = 1;  // thread 0: the workgroups that have started
  for (;;) {
    // here = 0 when the watchdog fires (a leader on its own waits for nobody, so it looks at the clock here)
    if (tid == 0) {
      if (here < (uint32_t)a.members) here = min(ld_sync(&a.ctl->ticket), (uint32_t)a.members);
      if (lv.tag % 64u == 0u && team_late(a, sm)) {
        team_fail(a, ERR_TIMEOUT);
        here = 0;
      }
    }
    const int32_t pos = lv.pos;
    const uint32_t v = team_level<G>(a, sm, lv, here);
    if (v == TEAM_STOP) {
      *stop = true;
      break;
    }
    if (lv.pos > pos) {  // the level had parents
      ++lev;
      *last = pos;
    }
    if (v != TEAM_ON) break;
  }
  *tag = lv.tag;
  *levels = lev;
  return lv.pos;
}

// The leader: the search and order of solo_matrix (engine_solo.hpp), a pass at a time.
template <class G>
__device__ __forceinline__ void team_lead(const TeamArgs& a, TeamSmem<G>& sm) {
  const int tid = threadIdx.x, ln = lane_id();
  const int32_t n = a.n;
  constexpr uint32_t kEpochs = 255;  // passes until the claims must be cleared again
  bool searching = a.mode != SOLO_RUN && a.start < 0 && n > 1, redo = false, stop = false;
  int32_t cur = a.start >= 0 ? a.start : n > 1 ? n / 2 : 0;
  int32_t iters = a.start < 0 && n == 1 ? 1 : 0, passes = 0, placed = n, lev = 0, last = 0;
  uint32_t tag = a.tag0, lastdist = 0, left = kEpochs;
  if (tid == 0) sm.due = SearchPasses{1u, 0u};
  while (searching || a.mode != SOLO_SEARCH) {
    if (searching && !redo) ++iters;
    const bool attempt = searching && !redo && a.mode == SOLO_ORDER && a.speculate > 0 && iters >= a.speculate;
    if (left == 0) {
      for (int32_t i = tid; i < n; i += G::T) st_sync(&a.claim[i], ~(uint64_t)0);
      left = kEpochs;
    }
    --left;
    if (tid == 0) {
      st_sync(&a.ctl->passes, (int32_t)sm.due.count);
      sm.deadline = min(sm.launch + a.budget_ticks * sm.due.count, wall_ticks() + a.budget_ticks);
      sm.t0 = sm.deadline - a.budget_ticks * sm.due.count;  // its own word moves the leader's deadline no further
      if (passes > 0) pass_beat(a.beat, sm.launch);
    }
    placed = team_pass<G>(a, sm, cur, searching && !attempt, left, &tag, &lev, &last, &stop);
    ++passes;
    if (placed != n || stop || !searching) break;
    if ((uint32_t)lev == lastdist) {  // cur is the start
      if (attempt || a.mode == SOLO_SEARCH) break;
      searching = false;
      if (tid == 0) ++sm.due.count;
      continue;
    }
    if (tid == 0) sm.due.sweep((uint32_t)lev, attempt);
    redo = attempt;  // a failed attempt is followed by the plain sweep from the same start
    if (redo) continue;
    lastdist = (uint32_t)lev;
    // the node of least row length among the last min(32, n - 1) of the last level, later ones winning ties. The last
    // level's queue entries are there: its members' words of what ended the pass -- a meeting of no parents, or a
    // redistribution of no children -- went out after them; a leader on its own waits for its stores here.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (wave_id() == 0) {
      const int32_t w = min(32, n - 1), p = n - w + ln;
      uint32_t key = ~0u;
      int32_t node = 0;
      if (ln < w && p >= last) {
        node = ld_sync(a.perm + p);
        key = ((uint32_t)(a.row_ptr[node + 1] - a.row_ptr[node]) << 6) | (uint32_t)(63 - ln);
      }
      const uint32_t best = wave_min(key);
      if (key == best) sm.cur = node;
    }
    __syncthreads();
    cur = sm.cur;
    __syncthreads();
  }
  if (tid == 0) {
    st_sync(&a.ctl->placed, (uint32_t)placed);
    st_sync(&a.ctl->nbatches, max(tag - a.tag0, 1u));
    st_sync(&a.ctl->start, cur);
    st_sync(&a.ctl->sweeps, iters);
    st_sync(&a.ctl->passes, passes);
    st_sync(&a.ctl->done, 1u);  // the others leave
  }
}

template <class G>
__global__ __launch_bounds__(G::T) void k_team(TeamArgs a) {
  using SM = TeamSmem<G>;
  RCM_LDS(SM, sm);
  const int tid = threadIdx.x;
  if (tid == 0) {
    sm.launch = sm.t0 = wall_ticks();
    sm.deadline = sm.t0 + a.budget_ticks;
    sm.g = (int32_t)atomic_add_u32(&a.ctl->ticket, 1u);
    sm.ckey[0] = ~0u;
    sm.lost = 0;
  }
  for (int i = tid; i < G::S; i += G::T) {
    sm.mark[i] = 0;
    sm.tab[i] = kNoSlot;
  }
  __syncthreads();
  if (sm.g >= a.members) return;
  if (sm.g == 0)
    team_lead<G>(a, sm);
  else
    team_help<G>(a, sm);
}

// Clears what a launch starts from: claims, the members' words, the control block; with tag0 0 the stages too (fresh
// memory, or entries of a launch that failed).
__global__ void k_team_init(TeamArgs a) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = t; i < a.n; i += stride) a.claim[i] = ~(uint64_t)0;
  for (int64_t i = t; i < (int64_t)kTeamMax * kTeamWordStride; i += stride) a.words[i] = 0ull;
  if (a.tag0 == 0)
    for (int64_t i = t; i < (int64_t)kTeamMax * a.cap * 2; i += stride) a.stage[0][i] = a.stage[1][i] = 0ull;
  if (t == 0) {
    Control c = {};
    *a.ctl = c;
  }
}

}  // namespace rcm
