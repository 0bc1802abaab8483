// bucket_csr.hpp -- device kernels that turn COO triples into a sorted, symmetrised CSR by buckets of consecutive rows.
//
// A sort of all entries on (row, column) by 8-bit digits passes over them once per digit, and the symmetrisation then
// sorts the transposes the same way and merges. Here every entry becomes one record, and its transpose another: the
// records are dealt to buckets of 2^sh rows in a pass or two, and each bucket is small enough to be sorted in the LDS of
// one workgroup. All that decides about a row of the result lies in its bucket: the entries (r, c) stored in it and the
// transposes of those stored as (c, r), so the parity of a pair is a count there, and no search in another row.
//
// A record is one word: row in the bucket, column, group, input index, from high to low. Its order is the order of the
// result (include/Graph.h:77-157, and the stable conversion after it): by row, column and insertion position; position
// follows the row that an entry is stored in, so the transposes (stored in row c) come before the row's own entries where
// c < r and after them where c > r -- the group bit -- and each of the two in input order. No two records are equal,
// so neither the deal nor the sort has to be stable.
//
// Dealing in one step writes single words: 4096 buckets, a 128-byte line each, are more than an XCD's cache keeps open, so
// most words leave it as a line of their own. From 128 buckets on it takes two steps, groups and then their buckets, and
// each step sorts a tile of records by bin in LDS first, so that they leave in runs. The values go along, so that the sort
// finds them in its bucket: gathered in input order, each costs a line.
// Measured on MI355X, the 128^3 stencil from its shuffled lower triangle (8.3M triples, 14.6M records, double values), us:
//   by digits and a merge               1700
//   one step, values gathered            634: count 46, deal 257, sort 331
//   two steps, values dealt              419: count 33, totals 22, deal 109 (350 MB), split 133 (470 MB), sort 117
#pragma once
#include "device_common.hpp"

namespace rcm_mx {
namespace {  // internal linkage: each library source that includes this has its own copy

// T threads a workgroup that sorts, TD one that counts or deals; CAP records (a power of two) and 2^ROWBITS rows a bucket
// at most; at most MAXB buckets. More than COARSE of them are dealt to in two steps, first to groups of 2^FB buckets.
template <int T_, int CAP_, int ROWBITS_, int MAXB_, int TD_, int FB_>
struct BucketGeo {
  static constexpr int T = T_, CAP = CAP_, ROWBITS = ROWBITS_, MAXB = MAXB_, TD = TD_, FB = FB_;
  static constexpr int EPT = CAP / T, NC = CAP / rcm::kWave;
  static constexpr int COARSE = MAXB >> FB;
  static constexpr int BINS = COARSE > (1 << FB) ? COARSE : 1 << FB;  // of one deal
  static constexpr int TILE = 4 * TD;                                 // records a deal holds at a time
  static_assert((CAP & (CAP - 1)) == 0 && CAP % T == 0 && T % rcm::kWave == 0 && NC <= T && CAP <= 65536, "geometry");
  static_assert(BINS <= TD && BINS <= 256, "a thread and a byte for a bin");
};

struct BucketJob {
  const int32_t* r;
  const int32_t* c;
  int64_t nnz;
  int64_t per;       // entries a workgroup counts and deals
  int32_t rows;
  int32_t buckets;
  int32_t groups;    // of 2^fb buckets
  int32_t sh;        // rows of a bucket, as a power of two
  int32_t fb;        // buckets of a group, as a power of two: 0 for a deal in one step
  int32_t col_bits, idx_bits;
  int32_t mirror;    // with the transposes
};

// Longest row that is ordered by counting; a bucket with a longer one is sorted as a whole.
constexpr uint32_t kBucketRank = 128;

template <class G>
struct CountSmem {
  uint32_t n[G::MAXB];
};

// table[w * buckets + b]: records of workgroup w in bucket b; group[g * workgroups + w]: in group g. *flag = ~0 for an
// index out of range.
template <class G>
__global__ __launch_bounds__(G::TD) void k_bucket_count(BucketJob J, uint32_t* table, uint32_t* group, uint32_t* flag) {
  using SM = CountSmem<G>;
  RCM_LDS(SM, sm);
  for (int b = threadIdx.x; b < J.buckets; b += G::TD) sm.n[b] = 0;
  __syncthreads();
  const int64_t e0 = (int64_t)blockIdx.x * J.per, e1 = e0 + J.per < J.nnz ? e0 + J.per : J.nnz;
  bool bad = false;
#pragma unroll 4
  for (int64_t k = e0 + threadIdx.x; k < e1; k += G::TD) {
    const int32_t a = J.r[k], b = J.c[k];
    if (a < 0 || a >= J.rows || b < 0 || b >= J.rows) {
      bad = true;
    } else {
      atomicAdd(&sm.n[a >> J.sh], 1u);
      if (J.mirror && a != b) atomicAdd(&sm.n[b >> J.sh], 1u);
    }
  }
  if (bad) *flag = ~0u;
  __syncthreads();
  for (int b = threadIdx.x; b < J.buckets; b += G::TD) table[(size_t)blockIdx.x * J.buckets + b] = sm.n[b];
  for (int g = threadIdx.x; g < J.groups; g += G::TD) {
    uint32_t n = 0;
    const int f = 1 << J.fb;
    for (int i = 0; i < f; ++i) {  // each thread from another of its buckets on: they lie in different banks
      const int b = (g << J.fb) + ((i + g) & (f - 1));
      n += b < J.buckets ? sm.n[b] : 0u;
    }
    group[(size_t)g * gridDim.x + blockIdx.x] = n;
  }
}

// base[b] = records of bucket b, to be scanned (base[buckets] = 0); *flag: the records of the largest, unless it is ~0.
__global__ __launch_bounds__(256) void k_bucket_total(const uint32_t* table, int32_t buckets, uint32_t wgs, uint32_t* base,
                                                     uint32_t* flag) {
  const int32_t b = (int32_t)(blockIdx.x * 256 + threadIdx.x);
  if (b > buckets) return;
  uint32_t n = 0;
  if (b < buckets) {
#pragma unroll 8
    for (uint32_t w = 0; w < wgs; ++w) n += table[(size_t)w * buckets + b];
    if (n > rcm::ld_sync(flag)) atomicMax(flag, n);
  }
  base[b] = n;
}

// cur[b] = base[b]: where the second step of a deal puts the next records.
__global__ __launch_bounds__(256) void k_bucket_cursors(const uint32_t* base, int32_t buckets, uint32_t* cur) {
  const int32_t b = (int32_t)(blockIdx.x * 256 + threadIdx.x);
  if (b < buckets) cur[b] = base[b];
}

template <class G, class V>
struct DealSmem {
  uint64_t rec[G::TILE];
  V val[G::TILE];
  uint8_t bin[G::TILE];
  uint32_t n[G::BINS];      // records of each bin in the tile
  uint32_t at[G::BINS];     // the first of them in the tile
  uint32_t to[G::BINS];     // where they go, less `at`
  uint32_t cur[G::BINS];    // where the workgroup's next records of a bin go (first step)
  uint32_t w[G::TD / rcm::kWave + 1];
};

// A tile of records, up to four to a thread (bin < 0: none), in LDS by bin, so that a bin's records leave in one run. A
// run starts at sm.cur[bin], which moves on, or with `cur` at that word, shared by all workgroups. Ends before a barrier.
template <class G, class V>
__device__ __forceinline__ void deal_tile(DealSmem<G, V>& sm, const uint64_t (&rec)[4], const V (&val)[4],
                                          const int (&bin)[4], int bins, uint32_t* cur, bool values, uint64_t* rec_out,
                                          V* val_out) {
  const int t = threadIdx.x;
  if (t < bins) sm.n[t] = 0;
  __syncthreads();
  uint32_t rank[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (bin[k] >= 0) rank[k] = atomicAdd(&sm.n[bin[k]], 1u);
  __syncthreads();
  const uint32_t n = t < bins ? sm.n[t] : 0u;
  uint32_t total;
  const uint32_t ex = rcm::block_excl_scan<G::TD>(n, sm.w, &total);
  if (t < bins) {
    uint32_t to = 0;
    if (cur) {
      if (n) to = atomicAdd(cur + t, n);
    } else {
      to = sm.cur[t];
      sm.cur[t] = to + n;
    }
    sm.at[t] = ex;
    sm.to[t] = to - ex;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (bin[k] < 0) continue;
    const uint32_t p = sm.at[bin[k]] + rank[k];
    sm.rec[p] = rec[k];
    sm.bin[p] = (uint8_t)bin[k];
    if (values) sm.val[p] = val[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t p = (uint32_t)(k * G::TD + t);
    if (p >= total) continue;
    const size_t o = (size_t)(sm.to[sm.bin[p]] + p);
    rec_out[o] = sm.rec[p];
    if (values) val_out[o] = sm.val[p];
  }
}

// First step: the records of workgroup w to their groups (buckets, where a group is one), behind those of the workgroups
// before it (group: k_bucket_count's, scanned). Values go along: gathered by the sort, in input order, they would cost a
// line each.
template <class G, class V>
__global__ __launch_bounds__(G::TD) void k_bucket_deal(BucketJob J, const uint32_t* group, const V* vals, uint64_t* rec_out,
                                                      V* val_out) {
  using SM = DealSmem<G, V>;
  RCM_LDS(SM, sm);
  const int t = threadIdx.x;
  if (t < J.groups) sm.cur[t] = group[(size_t)t * gridDim.x + blockIdx.x];
  const int64_t e0 = (int64_t)blockIdx.x * J.per, e1 = e0 + J.per < J.nnz ? e0 + J.per : J.nnz;
  const int gs = J.sh + J.fb;
  const uint32_t low = (uint32_t)(((uint64_t)1 << gs) - 1);
  for (int64_t k0 = e0; k0 < e1; k0 += 2 * G::TD) {
    uint64_t rec[4] = {};
    V val[4] = {};
    int bin[4] = {-1, -1, -1, -1};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t k = k0 + i * G::TD + t;
      if (k >= e1) continue;
      const uint32_t a = (uint32_t)J.r[k], b = (uint32_t)J.c[k];
      const uint32_t below = b < a ? 1u : 0u;
      // own entry: its group comes second where the column is below the row
      rec[i] = ((((uint64_t)(a & low) << J.col_bits | b) << 1 | below) << J.idx_bits) | (uint64_t)k;
      bin[i] = (int)(a >> gs);
      if (J.mirror && a != b) {  // in row b, column a: second where a > b, which is where `below` holds
        rec[2 + i] = ((((uint64_t)(b & low) << J.col_bits | a) << 1 | below) << J.idx_bits) | (uint64_t)k;
        bin[2 + i] = (int)(b >> gs);
      }
      if (vals) val[i] = val[2 + i] = vals[k];
    }
    deal_tile<G, V>(sm, rec, val, bin, J.groups, nullptr, vals != nullptr, rec_out, val_out);
    __syncthreads();
  }
}

// Second step: the records of a group, a tile at a time, to its buckets. Workgroup (g, j) of groups x `each`.
template <class G, class V>
__global__ __launch_bounds__(G::TD) void k_bucket_split(BucketJob J, const uint32_t* base, uint32_t* cur, int32_t each,
                                                       const uint64_t* rec_in, const V* val_in, uint64_t* rec_out,
                                                       V* val_out) {
  using SM = DealSmem<G, V>;
  RCM_LDS(SM, sm);
  const int t = threadIdx.x;
  const int32_t g = (int32_t)blockIdx.x / each, j = (int32_t)blockIdx.x % each;
  const int32_t b0 = g << J.fb, bins = min(1 << J.fb, J.buckets - b0);
  const uint32_t p0 = base[b0], p1 = base[b0 + bins];
  const int at = J.col_bits + 1 + J.idx_bits + J.sh;
  for (uint32_t q0 = p0 + (uint32_t)j * G::TILE; q0 < p1; q0 += (uint32_t)each * G::TILE) {
    uint64_t rec[4];
    V val[4] = {};
    int bin[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t q = q0 + (uint32_t)(k * G::TD + t);
      bin[k] = -1;
      if (q >= p1) continue;
      rec[k] = rec_in[q];
      bin[k] = (int)(rec[k] >> at);
      if (val_in) val[k] = val_in[q];
    }
    deal_tile<G, V>(sm, rec, val, bin, bins, cur + b0, val_in != nullptr, rec_out, val_out);
    __syncthreads();
  }
}

template <class G>
struct BucketSmem {
  uint64_t rec[G::CAP];
  uint16_t from[G::CAP];  // a record's place before the sort, for its value
  uint32_t off[(1 << G::ROWBITS) + 1];
  uint64_t keep[G::NC];   // per 64 records: those that stay
  uint32_t pre[G::NC];    // those before them
  uint32_t w[2 * (G::T / rcm::kWave) + 1];
  uint32_t drop;
};

// The first record in [a, b) that is not below v.
template <class SM>
__device__ __forceinline__ uint32_t bucket_lower(const SM& sm, uint32_t a, uint32_t b, uint64_t v) {
  while (a < b) {
    const uint32_t mid = (a + b) >> 1;
    if (sm.rec[mid] < v) a = mid + 1;
    else b = mid;
  }
  return a;
}

// One bucket: sorted, the transposes of evenly stored pairs taken out, and written as rows from the bucket's first record
// on (rp, ci, vout; with anything taken out these leave gaps, see k_bucket_close). kept[b]: its records that stay
// (kept[buckets] = 0). out[0] = 1: an evenly stored pair is not symmetric; out[1]: records taken out; out[2]:
// records.
// Bound by LDS and the latency of its phases, which three workgroups on a compute unit cover for each other.
template <class G, class V>
__global__ __launch_bounds__(G::T) void k_bucket_sort(BucketJob J, const uint32_t* base, const uint64_t* rec,
                                                     const V* vin, int32_t* rp, int32_t* ci, V* vout, uint32_t* kept,
                                                     uint32_t* out) {
  using SM = BucketSmem<G>;
  RCM_LDS(SM, sm);
  constexpr int T = G::T, EPT = G::EPT;
  const int t = threadIdx.x;
  const uint32_t b0 = base[blockIdx.x], m = base[blockIdx.x + 1] - b0;
  const int32_t row0 = (int32_t)(blockIdx.x << J.sh);
  const int nr = min(1 << J.sh, J.rows - row0);
  const int row_at = J.col_bits + 1 + J.idx_bits, key_at = J.idx_bits + 1;
  const uint32_t row_mask = (1u << J.sh) - 1u;  // above it: the bucket's place in its group
  for (int i = t; i <= nr; i += T) sm.off[i] = 0;
  if (t == 0) sm.drop = 0;
  uint64_t v[EPT];
  uint32_t to[EPT], from[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) v[k] = (uint32_t)(k * T + t) < m ? rec[(size_t)b0 + (uint32_t)(k * T + t)] : ~0ull;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < EPT; ++k)
    if ((uint32_t)(k * T + t) < m) to[k] = atomicAdd(&sm.off[(uint32_t)(v[k] >> row_at) & row_mask], 1u);
  __syncthreads();
  uint32_t longest = 0;
  for (int i0 = 0, carry = 0; i0 < nr; i0 += T) {
    const uint32_t l = i0 + t < nr ? sm.off[i0 + t] : 0u;
    uint32_t tot, mx;
    const uint32_t ex = rcm::block_excl_scan_max<T>(l, l, sm.w, &tot, &mx);
    if (i0 + t < nr) sm.off[i0 + t] = (uint32_t)carry + ex;
    carry += (int)tot;
    longest = max(longest, mx);
  }
  if (t == 0) sm.off[nr] = m;
  __syncthreads();
  if (longest <= kBucketRank) {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      if ((uint32_t)(k * T + t) >= m) continue;
      const uint32_t o = sm.off[(uint32_t)(v[k] >> row_at) & row_mask] + to[k];
      sm.rec[o] = v[k];
      sm.from[o] = (uint16_t)(k * T + t);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      if ((uint32_t)(k * T) >= m) break;
      const uint32_t i = (uint32_t)(k * T + t);
      if (i >= m) continue;
      v[k] = sm.rec[i];
      from[k] = sm.from[i];
      const uint32_t row = (uint32_t)(v[k] >> row_at) & row_mask, b = sm.off[row + 1];
      to[k] = sm.off[row];
      for (uint32_t q = sm.off[row]; q < b; ++q) to[k] += sm.rec[q] < v[k] ? 1u : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      if ((uint32_t)(k * T + t) >= m) continue;
      sm.rec[to[k]] = v[k];
      sm.from[to[k]] = (uint16_t)from[k];
    }
    __syncthreads();
  } else {  // a bitonic network over the next power of two
    uint32_t P = 1;
    while (P < m) P <<= 1;
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      sm.rec[k * T + t] = v[k];
      sm.from[k * T + t] = (uint16_t)(k * T + t);
    }
    __syncthreads();
    for (uint32_t s = 2; s <= P; s <<= 1)
      for (uint32_t d = s >> 1; d > 0; d >>= 1) {
        for (uint32_t i = (uint32_t)t; i < P / 2; i += T) {
          const uint32_t lo = 2 * i - (i & (d - 1)), hi = lo + d;
          const uint64_t x = sm.rec[lo], y = sm.rec[hi];
          if ((x > y) == ((lo & s) == 0)) {
            sm.rec[lo] = y;
            sm.rec[hi] = x;
            const uint16_t f = sm.from[lo];
            sm.from[lo] = sm.from[hi];
            sm.from[hi] = f;
          }
        }
        __syncthreads();
      }
  }
  // which records stay
  const uint32_t col_mask = (uint32_t)(((uint64_t)1 << J.col_bits) - 1);
  bool unsym = false, dropped = false;
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    if ((uint32_t)(k * T) >= m) break;
    const uint32_t i = (uint32_t)(k * T + t);
    bool stay = i < m;
    if (stay) {
      v[k] = sm.rec[i];
      const uint64_t key = v[k] >> key_at;
      if (J.mirror && ((i > 0 && sm.rec[i - 1] >> key_at == key) || (i + 1 < m && sm.rec[i + 1] >> key_at == key))) {
        const uint32_t row = (uint32_t)(key >> J.col_bits) & row_mask, r = (uint32_t)row0 + row, c = (uint32_t)key & col_mask;
        if (c != r) {
          const uint32_t a = sm.off[row], b = sm.off[row + 1];
          const uint32_t lo = bucket_lower(sm, a, b, key << key_at);
          const uint32_t hi = bucket_lower(sm, lo, b, (key + 1) << key_at);
          const uint32_t first = bucket_lower(sm, lo, hi, (key << key_at) + ((uint64_t)1 << J.idx_bits)) - lo;
          const uint32_t second = hi - lo - first;
          const bool odd = ((first + second) & 1u) != 0;
          const bool own = ((uint32_t)(v[k] >> J.idx_bits) & 1u) == (c < r ? 1u : 0u);
          stay = own || odd;
          unsym = unsym || (!odd && first != second);
        }
      }
      dropped = dropped || !stay;
    }
    const uint64_t bal = rcm::ballot(stay);
    if (rcm::lane_id() == 0) sm.keep[i / rcm::kWave] = bal;
  }
  if (unsym) out[0] = 1u;
  if (dropped) sm.drop = 1u;
  __syncthreads();
  const bool gaps = sm.drop != 0;
  uint32_t left = m;
  if (gaps) {
    const uint32_t n = (uint32_t)(t * rcm::kWave) < m ? (uint32_t)__popcll(sm.keep[t]) : 0u;
    const uint32_t ex = rcm::block_excl_scan<T>(n, sm.w, &left);
    if (t < G::NC) sm.pre[t] = ex;
    __syncthreads();
    if (t == 0) atomicAdd(out + 1, m - left);
  }
  const auto place = [&](uint32_t i) -> uint32_t {  // of record i among those that stay; i <= m
    if (!gaps) return i;
    if (i >= m) return left;
    const uint32_t g = i / rcm::kWave;
    return sm.pre[g] + (uint32_t)__popcll(sm.keep[g] & (((uint64_t)1 << (i % rcm::kWave)) - 1));
  };
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    if ((uint32_t)(k * T) >= m) break;
    const uint32_t i = (uint32_t)(k * T + t);
    if (i >= m) continue;
    if (gaps && ((sm.keep[i / rcm::kWave] >> (i % rcm::kWave)) & 1u) == 0) continue;
    const size_t o = (size_t)b0 + place(i);
    ci[o] = (int32_t)((uint32_t)(v[k] >> key_at) & col_mask);
    if (vin) vout[o] = vin[(size_t)b0 + sm.from[i]];
  }
  for (int i = t; i < nr; i += T) rp[row0 + i] = (int32_t)(b0 + place(sm.off[i]));
  if (t == 0) {
    kept[blockIdx.x] = left;
    if ((int32_t)blockIdx.x == J.buckets - 1) {
      kept[J.buckets] = 0;
      out[2] = b0 + m;
      rp[J.rows] = (int32_t)(b0 + left);
    }
  }
}

// Closes the gaps: bucket b's rows move from base[b] to the scanned kept[b].
template <class V>
__global__ __launch_bounds__(256) void k_bucket_close(BucketJob J, const uint32_t* base, const uint32_t* kept,
                                                     const int32_t* rp, const int32_t* ci, const V* v, int32_t* rp2,
                                                     int32_t* ci2, V* v2) {
  const uint32_t b0 = base[blockIdx.x], k0 = kept[blockIdx.x], n = kept[blockIdx.x + 1] - k0;
  for (uint32_t i = threadIdx.x; i < n; i += 256) {
    ci2[(size_t)k0 + i] = ci[(size_t)b0 + i];
    if (v) v2[(size_t)k0 + i] = v[(size_t)b0 + i];
  }
  const int32_t row0 = (int32_t)(blockIdx.x << J.sh);
  const int nr = min(1 << J.sh, J.rows - row0);
  for (int i = threadIdx.x; i < nr; i += 256) rp2[row0 + i] = (int32_t)((uint32_t)rp[row0 + i] - b0 + k0);
  if ((int32_t)blockIdx.x == J.buckets - 1 && threadIdx.x == 0) rp2[J.rows] = (int32_t)(k0 + n);
}

}  // namespace
}  // namespace rcm_mx
