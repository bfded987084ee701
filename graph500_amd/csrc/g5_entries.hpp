// g5_entries.hpp -- the directed entries of a graph on their way from tuples
// to sorted, deduplicated CSR rows (device kernels of g5_csr.hip).
//
// An entry is one uint64: a row-side id in the high word, a column-side id in
// the low word.  Every tuple a != b gives (a, b) and (b, a), so the entry set
// is symmetric and any pass may swap the two sides.  The passes:
//
//   k_partition    tuples -> entries grouped by ranges of their row-side id.
//                  Grouped entries make every per-vertex table access local:
//                  degrees are counted in LDS (k_bucket_degrees) instead of by
//                  2 m global atomics, and the lookups of new ids hit the L2.
//   k_partition    once or twice more, the column side relabelled and the
//                  row side turned into a position on the way.  The position
//                  of entry (r, c) among the sorted entries is estimated as
//                  P[r] + deg(r) * frac(c), P the degree prefix and frac(c)
//                  the share of all entries in columns below c: increasing in
//                  (r, c), in [P[r], P[r + 1]), and near the true rank,
//                  because the rows of a random graph share nearly one column
//                  distribution.  Grouped by L1 buckets: the rows whose P[r]
//                  falls into one stretch of W positions, whose sizes the
//                  degrees give exactly.
//   k_refine       each L1 bucket -> sub-buckets of 2^sub positions.
//   k_sort_sub     each sub-bucket in LDS: bin = position (about one entry
//                  each), rank within the bin by comparison, duplicates
//                  dropped, unique counts per row.
//   k_compact      the unique columns to their final place.
//
// Bytes per tuple: 12 + 16 written, then 16 + 16 three times, 16 + 8, 8 + 8:
// about 160 B, all of it in runs, against seven stable radix passes over
// 64-bit keys (24 B of traffic per entry and pass) plus two random id lookups
// and two random atomics per tuple.
#pragma once

#include "g5_prims.hpp"

namespace g5 {

constexpr int kPartThreads = 1024;
constexpr int kPartMax = 1024;  // buckets of one partition, one per thread
constexpr int kCursorPad = 8;   // a bucket cursor has a 64-byte line of its own

constexpr int kSubMax = 8192;     // sub-buckets of one L1 bucket
constexpr int kFracMax = 6401;    // entries of the column share table
constexpr int kDegVerts = 32768;  // vertices counted by one workgroup (128 KB of LDS)
constexpr int kDegBits = 28;      // low bits of a row word (k_row_words): its degree
constexpr uint64_t kDegMask = (UINT64_C(1) << kDegBits) - 1;

// info words of a build
enum { I_SUBS = 0, I_WIDE, I_OVERFLOW, I_MAXDEG, I_ACTIVE, I_LOOPS, I_NUM };

// Inclusive scan over a wave, 32-bit.
__device__ __forceinline__ uint32_t wave_incl_scan32(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// Exclusive scan of one value per thread over a block of kThreads; s_w holds
// kThreads / 64 words.  Ends with a barrier.
template <int kThreads>
__device__ __forceinline__ uint32_t block_excl_scan32(uint32_t v, uint32_t* s_w, uint32_t& tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t inc = wave_incl_scan32(v);
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  uint32_t off = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {
    const uint32_t x = s_w[w];
    off += (w < wave) ? x : 0;
    all += x;
  }
  __syncthreads();
  tot = all;
  return off + inc - v;
}

// --- the position estimate ---

// Share of all entries in columns below c, as a 32-bit fraction: linear
// between samples of P.  Degree order (flat = -1): 256 samples per octave of
// c, exact for the 256 top hubs, dense where the degrees fall fast.  Other
// orders: samples 2^flat columns apart.
struct FracMap {
  static __host__ __device__ uint32_t index(uint32_t c, int flat, int& sh) {
    if (flat >= 0) {
      sh = flat;
      return c >> flat;
    }
    sh = 0;
    if (c < 256) return c;
    const int e = 31 - __builtin_clz(c);
    sh = e - 8;
    return ((uint32_t)(e - 7) << 8) + ((c >> sh) & 255);
  }
  // first column of sample i
  static __host__ __device__ uint64_t start(uint32_t i, int flat) {
    if (flat >= 0) return (uint64_t)i << flat;
    if (i < 256) return i;
    return (uint64_t)(256 + (i & 255)) << ((i >> 8) - 1);
  }
  static __device__ uint32_t at(const uint32_t* f, uint32_t c, int flat) {
    int sh;
    const uint32_t i = index(c, flat, sh);
    const uint32_t f0 = f[i];
    const uint32_t low = c & (uint32_t)((UINT64_C(1) << sh) - 1);
    return f0 + (uint32_t)(((uint64_t)(f[i + 1] - f0) * low) >> sh);
  }
};

__global__ void k_frac_table(const uint64_t* __restrict__ P, int64_t rows, int flat, int count,
                             uint32_t* __restrict__ f) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const uint64_t s = FracMap::start((uint32_t)i, flat);
  const double x = (double)P[(int64_t)s < rows ? (int64_t)s : rows] / (double)P[rows] * 4294967296.0;
  f[i] = x < 4294967295.0 ? (uint32_t)x : 0xFFFFFFFFu;
}

// Per original id: new id, and the row word P[row] << kDegBits | degree that
// the position estimate of its entries needs in one lookup (degrees beyond
// the field are cut, which keeps the estimate below the next row's first).
__global__ void k_row_words(const uint32_t* __restrict__ new2old, int64_t n, const uint64_t* __restrict__ P,
                            int64_t rows, uint32_t* __restrict__ old2new, uint64_t* __restrict__ row_word) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t o = new2old[v];
    old2new[o] = (uint32_t)v;
    if (v < rows) {
      const uint64_t p = P[v], d = P[v + 1] - p;
      row_word[o] = (p << kDegBits) | (d < kDegMask ? d : kDegMask);
    }
  }
}

// --- sources of a partition: kPer entries per thread and tile.  raw() only
// starts the loads, so that a tile's are in flight while the previous tile is
// written; finish() makes the entries. ---

// Tuples (ids below 2^32) in both directions, by ranges of 2^shift ids; loops
// are counted per vertex and dropped.
struct SrcTuples {
  static constexpr int kPer = 12, kRaw = 6, kTile = kPer * kPartThreads;
  static constexpr bool kKeep = false;  // the bucket follows from the entry
  const g5_packed_edge* e;
  int64_t m;
  uint32_t* loops;
  int shift;
  __host__ int64_t tiles() const { return (m + kTile / 2 - 1) / (kTile / 2); }
  __device__ void stage() const {}
  __device__ uint32_t bucket_of(uint64_t x) const { return (uint32_t)(x >> 32) >> shift; }
  __device__ void raw(int64_t tile, uint64_t (&r)[kRaw]) const {
#pragma unroll
    for (int j = 0; j < kRaw; ++j) {
      const int64_t i = tile * (kTile / 2) + j * kPartThreads + threadIdx.x;
      r[j] = 0;
      if (i < m) r[j] = ((uint64_t)e[i].v0_low << 32) | e[i].v1_low;
    }
  }
  __device__ void finish(int64_t tile, const uint64_t (&r)[kRaw], uint64_t (&out)[kPer], uint32_t (&b)[kPer],
                         uint32_t& ok) const {
    ok = 0;
#pragma unroll
    for (int j = 0; j < kRaw; ++j) {
      const int64_t i = tile * (kTile / 2) + j * kPartThreads + threadIdx.x;
      const uint32_t x = (uint32_t)(r[j] >> 32), y = (uint32_t)r[j];
      if (i < m) {
        if (x == y) atomicAdd(&loops[x], 1u);
        else ok |= 3u << (2 * j);
      }
      out[2 * j] = r[j];
      out[2 * j + 1] = ((uint64_t)y << 32) | x;
      b[2 * j] = x >> shift;
      b[2 * j + 1] = y >> shift;
    }
  }
};

// Entries (x, y) as (y, new id of x), by ranges of y.
struct SrcRelabel {
  static constexpr int kPer = 12, kRaw = 12, kTile = kPer * kPartThreads;
  static constexpr bool kKeep = false;
  const uint64_t* in;
  int64_t n;
  const uint32_t* old2new;
  int shift;
  __host__ int64_t tiles() const { return (n + kTile - 1) / kTile; }
  __device__ void stage() const {}
  __device__ uint32_t bucket_of(uint64_t x) const { return (uint32_t)(x >> 32) >> shift; }
  __device__ void raw(int64_t tile, uint64_t (&r)[kRaw]) const {
#pragma unroll
    for (int j = 0; j < kRaw; ++j) {
      const int64_t i = tile * kTile + j * kPartThreads + threadIdx.x;
      r[j] = i < n ? in[i] : 0;
    }
  }
  __device__ void finish(int64_t tile, const uint64_t (&r)[kRaw], uint64_t (&out)[kPer], uint32_t (&b)[kPer],
                         uint32_t& ok) const {
    ok = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int64_t i = tile * kTile + j * kPartThreads + threadIdx.x;
      const uint32_t y = (uint32_t)r[j];
      out[j] = (uint64_t)y << 32;
      b[j] = y >> shift;
      if (i < n) {
        ok |= 1u << j;
        out[j] |= old2new[r[j] >> 32];
      }
    }
  }
};

// Entries (x, y) as (position in the L1 bucket, column), by L1 buckets: x an
// original id, y the column's new id or, with kBoth, its original id.
template <bool kBoth>
struct SrcPosition {
  static constexpr int kPer = 6, kRaw = 6, kTile = kPer * kPartThreads;
  static constexpr bool kKeep = true;
  const uint64_t* in;
  int64_t n;
  const uint32_t* old2new;
  const uint64_t* row_word;
  const uint64_t* base;  // first position of every L1 bucket
  int nb1, wshift;
  const uint32_t* frac;
  int frac_count, flat;
  __host__ int64_t tiles() const { return (n + kTile - 1) / kTile; }
  __device__ uint32_t* lds_frac() const {
    __shared__ uint32_t s_f[kFracMax];
    return s_f;
  }
  __device__ uint64_t* lds_base() const {
    __shared__ uint64_t s_base[kPartMax];
    return s_base;
  }
  __device__ void stage() const {
    for (int i = threadIdx.x; i < frac_count; i += kPartThreads) lds_frac()[i] = frac[i];
    for (int i = threadIdx.x; i < nb1; i += kPartThreads) lds_base()[i] = base[i];
  }
  __device__ uint32_t bucket_of(uint64_t) const { return 0; }
  __device__ void raw(int64_t tile, uint64_t (&r)[kRaw]) const {
#pragma unroll
    for (int j = 0; j < kRaw; ++j) {
      const int64_t i = tile * kTile + j * kPartThreads + threadIdx.x;
      r[j] = i < n ? in[i] : 0;
    }
  }
  __device__ void finish(int64_t tile, const uint64_t (&r)[kRaw], uint64_t (&out)[kPer], uint32_t (&b)[kPer],
                         uint32_t& ok) const {
    ok = 0;
    constexpr int kHalf = kPer / 2;  // lookups in flight per thread; twelve entries per thread spill and are slower
#pragma unroll
    for (int h = 0; h < kPer; h += kHalf) {
      uint64_t w[kHalf];
      uint32_t c[kHalf];
#pragma unroll
      for (int k = 0; k < kHalf; ++k) {
        const int j = h + k;
        const int64_t i = tile * kTile + j * kPartThreads + threadIdx.x;
        w[k] = 0;
        c[k] = (uint32_t)r[j];
        if (i < n) {
          ok |= 1u << j;
          w[k] = row_word[r[j] >> 32];
          if (kBoth) c[k] = old2new[c[k]];
        }
      }
#pragma unroll
      for (int k = 0; k < kHalf; ++k) {
        const int j = h + k;
        const uint64_t p = w[k] >> kDegBits, d = w[k] & kDegMask;
        b[j] = (uint32_t)(p >> wshift);
        const uint32_t q = (uint32_t)(p - lds_base()[b[j]]) + (uint32_t)((d * FracMap::at(lds_frac(), c[k], flat)) >> 32);
        out[j] = ((uint64_t)q << 32) | c[k];
      }
    }
  }
};

// One pass: a workgroup ranks a tile's entries by bucket with LDS atomics
// (the order inside a bucket does not matter), reserves every bucket's run
// with one atomic on its cursor, places the entries bucket by bucket in LDS
// and writes the runs.  cursor[i * kCursorPad] starts at bucket i's first
// output index; the caller made the buckets' sizes exact.  One workgroup of
// 16 waves per CU: what bounds the pass is the length of the runs (a run's
// first and last line are shared with another workgroup, often on another
// XCD, and reach memory in parts), so the tile takes most of the LDS.
template <class Src>
__global__ void __launch_bounds__(kPartThreads) k_partition(Src src, int64_t tiles,
                                                            unsigned long long* __restrict__ cursor,
                                                            uint64_t* __restrict__ out) {
  constexpr int kPer = Src::kPer;
  __shared__ uint64_t s_e[Src::kTile];
  __shared__ uint64_t s_dst[kPartMax];
  __shared__ uint32_t s_cnt[kPartMax];
  __shared__ uint32_t s_w[kPartThreads / 64];
  __shared__ uint16_t s_b[Src::kKeep ? Src::kTile : 1];
  static_assert(kPartMax == kPartThreads, "one bucket per thread");
  const int t = threadIdx.x;
  src.stage();
  s_cnt[t] = 0;
  uint64_t raw[Src::kRaw];
  if ((int64_t)blockIdx.x < tiles) src.raw(blockIdx.x, raw);
  __syncthreads();
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    uint64_t e[kPer];
    uint32_t b[kPer], ok;
    src.finish(tile, raw, e, b, ok);
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if ((ok >> j) & 1) b[j] = (b[j] << 16) | atomicAdd(&s_cnt[b[j]], 1u);
    __syncthreads();
    const uint32_t c = s_cnt[t];
    uint32_t total;
    const uint32_t x = block_excl_scan32<kPartThreads>(c, s_w, total);
    if (c) s_dst[t] = atomicAdd(cursor + t * kCursorPad, (unsigned long long)c) - x;
    s_cnt[t] = x;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if ((ok >> j) & 1) {
        const uint32_t p = s_cnt[b[j] >> 16] + (b[j] & 0xFFFF);
        s_e[p] = e[j];
        if (Src::kKeep) s_b[p] = (uint16_t)(b[j] >> 16);
      }
    if (tile + gridDim.x < tiles) src.raw(tile + gridDim.x, raw);
    __syncthreads();
    for (uint32_t p = t; p < total; p += kPartThreads) {
      const uint64_t v = s_e[p];
      out[s_dst[Src::kKeep ? s_b[p] : src.bucket_of(v)] + p] = v;
    }
    s_cnt[t] = 0;
    __syncthreads();
  }
}

// Entries per range of 2^shift ids and the number of loops.
__global__ void __launch_bounds__(kBlock) k_part_count(const g5_packed_edge* __restrict__ e, int64_t m, int shift,
                                                       int nb, unsigned long long* __restrict__ counts,
                                                       unsigned long long* __restrict__ info) {
  __shared__ uint32_t s[kPartMax];
  __shared__ uint64_t s_wave[kBlock / 64];
  for (int i = threadIdx.x; i < nb; i += kBlock) s[i] = 0;
  __syncthreads();
  uint64_t loops = 0;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
#pragma unroll 4
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < m; i += stride) {
    const uint32_t a = e[i].v0_low, b = e[i].v1_low;
    if (a == b) {
      ++loops;
    } else {
      atomicAdd(&s[a >> shift], 1u);
      atomicAdd(&s[b >> shift], 1u);
    }
  }
  loops = wave_sum(loops);
  if ((threadIdx.x & 63) == 0) s_wave[threadIdx.x >> 6] = loops;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t l = 0;
    for (int w = 0; w < kBlock / 64; ++w) l += s_wave[w];
    if (l) atomicAdd(info + I_LOOPS, (unsigned long long)l);
  }
  for (int i = threadIdx.x; i < nb; i += kBlock)
    if (s[i]) atomicAdd(counts + i * kCursorPad, (unsigned long long)s[i]);
}

// counts -> first index of every bucket, kept in off[0, nb] and written to the
// cursors of both partitions over the same ranges (one workgroup).
__global__ void __launch_bounds__(kPartMax) k_part_offsets(const unsigned long long* __restrict__ counts, int nb,
                                                           uint64_t* __restrict__ off,
                                                           unsigned long long* __restrict__ cursor0,
                                                           unsigned long long* __restrict__ cursor1) {
  __shared__ uint64_t s_wave[kPartMax / 64];
  const int t = threadIdx.x;
  const uint64_t v = t < nb ? counts[t * kCursorPad] : 0;
  const uint64_t inc = wave_incl_scan(v);
  if ((t & 63) == 63) s_wave[t >> 6] = inc;
  __syncthreads();
  uint64_t base = 0;
  for (int w = 0; w < (t >> 6); ++w) base += s_wave[w];
  const uint64_t pre = base + inc - v;
  if (t < nb) {
    off[t] = pre;
    cursor0[t * kCursorPad] = pre;
    cursor1[t * kCursorPad] = pre;
    if (t == nb - 1) off[nb] = pre + v;
  }
}

// f(entry) for the entries [at, end) by a workgroup of 1024, kEachLoads
// 16-byte loads in flight per thread.
constexpr int kEachLoads = 4;
template <class F>
__device__ __forceinline__ void each_entry(const uint64_t* __restrict__ in, uint64_t at, uint64_t end, F f) {
  constexpr int kBatch = 1024 * 2 * kEachLoads;
  const int t = threadIdx.x;
  if ((at & 1) && at < end) {  // to a 16-byte boundary
    if (t == 0) f(in[at]);
    ++at;
  }
  for (; at + kBatch <= end; at += kBatch) {
    const ulonglong2* p = (const ulonglong2*)(in + at) + t;
    ulonglong2 e[kEachLoads];
#pragma unroll
    for (int j = 0; j < kEachLoads; ++j) e[j] = p[j * 1024];
#pragma unroll
    for (int j = 0; j < kEachLoads; ++j) {
      f(e[j].x);
      f(e[j].y);
    }
  }
#pragma unroll 4
  for (at += t; at < end; at += 1024) f(in[at]);
}

// Degrees (duplicates counted) of the vertices [base, base + 2^sub_shift):
// their bucket's entries counted in LDS.  A bucket of more than kDegVerts
// vertices takes several workgroups, each reading the whole bucket; 8 apart
// in the grid, they run on one XCD at the same time and all but the first
// find the entries in its L2 (there are 1024 buckets then, a multiple of 8).
// Bound by the loads in flight: with 128 KB of LDS there are 16 waves on a CU,
// so a thread has four 16-byte loads under way.  Against one 8-byte load after
// another and the parts of a bucket next to each other in the grid: SCALE 18
// 67 -> 56 us, 22 0.56 -> 0.36 ms, 25 2.94 -> 1.71 ms (5.0 TB/s), 26 (2 parts)
// 9.6 -> 3.6 ms, 28 (8 parts) 131.6 -> 31.7 ms (17 TB/s out of the L2; 83 ms
// with the parts next to each other, 36 ms with 8 loads, 33 ms with 16).
__global__ void __launch_bounds__(1024) k_bucket_degrees(const uint64_t* __restrict__ in,
                                                         const uint64_t* __restrict__ off, int shift, int sub_shift,
                                                         int64_t n, uint32_t* __restrict__ deg,
                                                         unsigned long long* __restrict__ info) {
  __shared__ uint32_t s[kDegVerts];
  __shared__ uint32_t s_red[2];
  const int t = threadIdx.x;
  const int parts = shift - sub_shift;  // log2 of the workgroups per bucket
  uint32_t bucket = blockIdx.x, part = 0;
  if (parts) {
    bucket = (blockIdx.x >> (3 + parts) << 3) + (blockIdx.x & 7);
    part = blockIdx.x >> 3 & ((1u << parts) - 1);
  }
  const uint32_t width = 1u << sub_shift;
  const uint32_t base = (bucket << shift) + (part << sub_shift);
  for (uint32_t i = t; i < width; i += 1024) s[i] = 0;
  if (t < 2) s_red[t] = 0;
  __syncthreads();
  each_entry(in, off[bucket], off[bucket + 1], [&](uint64_t e) {
    const uint32_t d = (uint32_t)(e >> 32) - base;
    if (d < width) atomicAdd(&s[d], 1u);
  });
  __syncthreads();
  uint32_t mx = 0, act = 0;
  for (uint32_t i = t; i < width; i += 1024) {
    if ((int64_t)base + i >= n) break;
    const uint32_t d = s[i];
    deg[base + i] = d;
    mx = d > mx ? d : mx;
    act += d != 0;
  }
  if (mx) atomicMax(&s_red[0], mx);
  if (act) atomicAdd(&s_red[1], act);
  __syncthreads();
  if (t == 0 && s_red[1]) {
    atomicMax(info + I_MAXDEG, (unsigned long long)s_red[0]);
    atomicAdd(info + I_ACTIVE, (unsigned long long)s_red[1]);
  }
}

// L1 buckets: rows [bound[i], bound[i + 1]), the rows whose first position
// lies in [i 2^wshift, (i + 1) 2^wshift); base = that first position, sub0 =
// the first sub-bucket (one workgroup, nb1 <= kPartMax).
__global__ void __launch_bounds__(kPartMax) k_l1_setup(const uint64_t* __restrict__ P, int64_t rows, int wshift,
                                                       int sub, int nb1, uint64_t* __restrict__ base,
                                                       uint32_t* __restrict__ sub0,
                                                       unsigned long long* __restrict__ cursor,
                                                       uint64_t* __restrict__ sub_pos,
                                                       unsigned long long* __restrict__ info) {
  __shared__ uint64_t s_base[kPartMax + 1];
  __shared__ uint32_t s_w[kPartMax / 64];
  const int t = threadIdx.x;
  if (t < nb1) {
    const uint64_t key = (uint64_t)t << wshift;
    int64_t lo = 0, hi = rows;  // first row with P >= key
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (P[mid] < key) lo = mid + 1; else hi = mid;
    }
    s_base[t] = P[lo];
  }
  if (t == 0) s_base[nb1] = P[rows];
  __syncthreads();
  uint32_t nsub = 0;
  if (t < nb1) {
    const uint64_t subs = (s_base[t + 1] - s_base[t] + (UINT64_C(1) << sub) - 1) >> sub;
    if (subs > kSubMax) atomicOr(info + I_WIDE, 1ull);
    nsub = (uint32_t)(subs > kSubMax ? kSubMax : subs);
  }
  uint32_t total;
  const uint32_t first = block_excl_scan32<kPartMax>(nsub, s_w, total);
  if (t < nb1) {
    base[t] = s_base[t];
    sub0[t] = first;
    cursor[t * kCursorPad] = s_base[t];
  }
  if (t == 0) {
    base[nb1] = s_base[nb1];
    sub0[nb1] = total;
    sub_pos[total] = s_base[nb1];
    info[I_SUBS] = total;
  }
}

// The row that owns every sub-bucket's first position.
__global__ void __launch_bounds__(kBlock) k_sub_rows(const uint64_t* __restrict__ P, int64_t rows, int wshift, int sub,
                                                     const uint64_t* __restrict__ base,
                                                     const uint32_t* __restrict__ sub0,
                                                     const unsigned long long* __restrict__ info,
                                                     uint32_t* __restrict__ sub_row) {
  if (info[I_WIDE]) return;
  const uint64_t round = (UINT64_C(1) << sub) - 1;
  for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (int64_t)gridDim.x * kBlock) {
    const uint64_t p0 = P[r], p1 = P[r + 1];
    if (p0 == p1) continue;
    const uint32_t i = (uint32_t)(p0 >> wshift);
    const uint64_t b = base[i], end = p1 - b;
    for (uint64_t j = (p0 - b + round) >> sub; (j << sub) < end; ++j) sub_row[sub0[i] + j] = (uint32_t)r;
  }
}

// One workgroup per L1 bucket: counts its sub-buckets in LDS, then moves its
// entries there tile by tile like k_partition, with the cursors in registers
// (thread t's consecutive sub-buckets): no other workgroup writes them.
// Counted by 16-byte loads (each_entry) instead of 8-byte ones: SCALE 18
// 89 -> 78 us, 25 7.4 -> 6.8 ms (3.8 TB/s), 27 26.5 -> 23.7 ms.
constexpr int kRefinePer = 11;
constexpr int kRefineTile = 1024 * kRefinePer;
__global__ void __launch_bounds__(1024) k_refine(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, int sub,
                                                 const uint64_t* __restrict__ base, const uint32_t* __restrict__ sub0,
                                                 uint64_t* __restrict__ sub_pos, uint64_t* __restrict__ sub_off,
                                                 uint32_t* __restrict__ sub_cnt,
                                                 const unsigned long long* __restrict__ info) {
  __shared__ uint64_t s_e[kRefineTile];
  __shared__ uint32_t s_cnt[kSubMax];
  __shared__ uint32_t s_dst[kSubMax];
  __shared__ uint32_t s_w[1024 / 64];
  if (info[I_WIDE]) return;
  const int t = threadIdx.x, sh = 32 + sub;
  const uint64_t b0 = base[blockIdx.x], b1 = base[blockIdx.x + 1];
  const uint32_t first = sub0[blockIdx.x];
  const int nsub = (int)(sub0[blockIdx.x + 1] - first);
  if (nsub == 0) return;
  const int own = (nsub + 1023) / 1024, sb0 = t * own;  // this thread's sub-buckets
  constexpr int kOwn = kSubMax / 1024;
  for (int i = t; i < nsub; i += 1024) s_cnt[i] = 0;
  __syncthreads();
  each_entry(in, b0, b1, [&](uint64_t e) { atomicAdd(&s_cnt[e >> sh], 1u); });
  __syncthreads();
  uint32_t cur[kOwn], sum = 0, total;
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    cur[j] = j < own && sb0 + j < nsub ? s_cnt[sb0 + j] : 0;
    sum += cur[j];
  }
  uint32_t run = block_excl_scan32<1024>(sum, s_w, total);
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const uint32_t c = cur[j];
    cur[j] = run;
    if (j < own && sb0 + j < nsub) {
      const uint32_t sb = first + sb0 + j;
      sub_pos[sb] = b0 + ((uint64_t)(sb0 + j) << sub);
      sub_off[sb] = b0 + run;
      sub_cnt[sb] = c;
      s_cnt[sb0 + j] = 0;
    }
    run += c;
  }
  uint64_t raw[kRefinePer];
#pragma unroll
  for (int j = 0; j < kRefinePer; ++j) {
    const uint64_t i = b0 + j * 1024 + t;
    raw[j] = i < b1 ? in[i] : 0;
  }
  __syncthreads();
  for (uint64_t at = b0; at < b1; at += kRefineTile) {
    uint32_t r[kRefinePer];
#pragma unroll
    for (int j = 0; j < kRefinePer; ++j)
      if (at + j * 1024 + t < b1) r[j] = atomicAdd(&s_cnt[raw[j] >> sh], 1u);
    __syncthreads();
    uint32_t c[kOwn];
    sum = 0;
#pragma unroll
    for (int j = 0; j < kOwn; ++j) {
      c[j] = j < own && sb0 + j < nsub ? s_cnt[sb0 + j] : 0;
      sum += c[j];
    }
    run = block_excl_scan32<1024>(sum, s_w, total);
#pragma unroll
    for (int j = 0; j < kOwn; ++j) {
      if (j < own && sb0 + j < nsub) {
        s_cnt[sb0 + j] = run;
        s_dst[sb0 + j] = cur[j] - run;
      }
      run += c[j];
      cur[j] += c[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRefinePer; ++j)
      if (at + j * 1024 + t < b1) s_e[s_cnt[raw[j] >> sh] + r[j]] = raw[j];
#pragma unroll
    for (int j = 0; j < kRefinePer; ++j) {
      const uint64_t i = at + kRefineTile + j * 1024 + t;
      raw[j] = i < b1 ? in[i] : 0;
    }
    __syncthreads();
    for (uint32_t p = t; p < total; p += 1024) {
      const uint64_t v = s_e[p];
      out[b0 + (uint32_t)(s_dst[v >> sh] + p)] = v;
    }
#pragma unroll
    for (int j = 0; j < kOwn; ++j)
      if (j < own && sb0 + j < nsub) s_cnt[sb0 + j] = 0;
    __syncthreads();
  }
}

typedef uint16_t half_word __attribute__((may_alias));  // bins are counted by pairs, read one by one

// One workgroup per sub-bucket: its entries sorted by (position, column) in
// LDS and deduplicated; the unique columns replace the entries in place (as
// uint32 from the sub-bucket's first byte on).  A bin is one position, so the
// entries of a bin share a row and are ranked by column alone; the bins hold
// about one entry each, so the ranking takes a couple of LDS reads per entry.
// Unique counts per row: a stored value for a row that lies inside the
// sub-bucket, an atomic add for the rows that cross its ends.  A sub-bucket
// may hold twice its positions; the register bound keeps at least four
// workgroups of 2^11 positions per CU (the compiler's own choice left one).
// Bound by LDS operations, so neighbouring lanes take neighbouring words: the
// bins are 16-bit counts, eight in one uint4 a thread, and places are numbered
// by groups of 64 (a ballot and a scan of the groups).  With 32-bit bins and
// sixteen consecutive places a thread, 8 and 16 lanes met in a bank: SCALE 20
// 221 -> 183 us, 22 0.82 -> 0.66 ms, 25 6.42 -> 5.03 ms (2.6 TB/s), 27 30.9 ->
// 25.6 ms.  Ranking two or four entries of a thread at once: 2 % slower.
template <int kSub>
struct SubSort {
  static constexpr int kWidth = 1 << kSub, kCap = 2 * kWidth, kPer = 16, kThreads = kCap / kPer;
};
template <int kSub>
__global__ void __launch_bounds__(SubSort<kSub>::kThreads, 4)
    k_sort_sub(uint64_t* __restrict__ x, const uint64_t* __restrict__ sub_off, const uint32_t* __restrict__ sub_cnt,
               const uint64_t* __restrict__ sub_pos, const uint32_t* __restrict__ sub_row,
               const uint64_t* __restrict__ P, int64_t rows, uint32_t* __restrict__ row_unique,
               uint32_t* __restrict__ sub_unique, unsigned long long* __restrict__ info) {
  constexpr int kWidth = SubSort<kSub>::kWidth, kCap = SubSort<kSub>::kCap, kPer = SubSort<kSub>::kPer;
  constexpr int kThreads = SubSort<kSub>::kThreads;
  constexpr int kBins = kWidth / kThreads;  // bins per thread in the scan
  constexpr int kGroups = kCap / 64;
  __shared__ uint32_t s_g[kGroups];
  __shared__ uint32_t s_col[kCap];
  __shared__ uint4 s_bins[kWidth / 8 + 1];  // entries per bin, then first places: 16 bits each
  half_word* const s_start = reinterpret_cast<half_word*>(s_bins);
  uint32_t* const s_pair = reinterpret_cast<uint32_t*>(s_bins);
  __shared__ uint16_t s_up[kCap + 1];  // unique flags, then unique entries before a place
  __shared__ uint32_t s_w[kThreads / 64];
  const uint32_t sub = blockIdx.x;
  const int t = threadIdx.x;
  const bool in_range = !info[I_WIDE] && sub < info[I_SUBS];
  const uint32_t cnt = in_range ? sub_cnt[sub] : 0;
  if (!in_range || cnt > (uint32_t)kCap) {
    if (t == 0) {
      sub_unique[sub] = 0;
      if (in_range) atomicOr(info + I_OVERFLOW, 1ull);
    }
    return;
  }
  const uint64_t off = sub_off[sub], pos = sub_pos[sub], pos_end = sub_pos[sub + 1];
  const int64_t row0 = sub_row[sub];
  static_assert(kBins == 8, "a thread's bins are one uint4");
  s_bins[t] = uint4{0, 0, 0, 0};
  __syncthreads();
  uint32_t col[kPer], br[kPer];  // bin << 16 | arrival in the bin
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint32_t i = j * kThreads + t;
    const uint64_t e = i < cnt ? x[off + i] : 0;
    col[j] = (uint32_t)e;
    br[j] = (uint32_t)(e >> 32) & (kWidth - 1);
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if ((uint32_t)(j * kThreads + t) < cnt) {
      const uint32_t at = br[j] & 1 ? 16 : 0, old = atomicAdd(&s_pair[br[j] >> 1], 1u << at);
      br[j] = (br[j] << 16) | (old >> at & 0xFFFF);
    }
  __syncthreads();
  {
    const uint4 c = s_bins[t];
    uint32_t w[4] = {c.x, c.y, c.z, c.w}, sum = 0, total;
#pragma unroll
    for (int j = 0; j < 4; ++j) sum += (w[j] & 0xFFFF) + (w[j] >> 16);
    uint32_t run = block_excl_scan32<kThreads>(sum, s_w, total);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t odd = run + (w[j] & 0xFFFF), next = odd + (w[j] >> 16);
      w[j] = run | odd << 16;
      run = next;
    }
    s_bins[t] = uint4{w[0], w[1], w[2], w[3]};
    if (t == 0) s_start[kWidth] = (half_word)cnt;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if ((uint32_t)(j * kThreads + t) < cnt) s_col[s_start[br[j] >> 16] + (br[j] & 0xFFFF)] = col[j];
  __syncthreads();
  // rank within the bin: smaller columns, then equal ones that came earlier
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if ((uint32_t)(j * kThreads + t) < cnt) {
      const uint32_t bin = br[j] >> 16, lo = s_start[bin], hi = s_start[bin + 1], own = lo + (br[j] & 0xFFFF);
      uint32_t less = 0, before = 0;
#pragma unroll 1
      for (uint32_t k = lo; k < hi; ++k) {
        const uint32_t c = s_col[k];
        less += c < col[j];
        before += c == col[j] && k < own;
      }
      br[j] = ((lo + less + before) << 1) | (before == 0);
    }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if ((uint32_t)(j * kThreads + t) < cnt) {
      s_col[br[j] >> 1] = col[j];
      s_up[br[j] >> 1] = (uint16_t)(br[j] & 1);
    }
  __syncthreads();
  // unique entries before every place, counted by groups of 64 places
  uint32_t flags = 0, total = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint32_t p = j * kThreads + t;
    const bool u = p < cnt && s_up[p];
    if (u) {
      col[j] = s_col[p];
      flags |= 1u << j;
    }
    const uint64_t m = __ballot(u);
    br[j] = __popcll(m & ((UINT64_C(1) << (t & 63)) - 1));
    if ((t & 63) == 0) s_g[p >> 6] = (uint32_t)__popcll(m);
  }
  __syncthreads();
  {
    const uint32_t v = t < kGroups ? s_g[t] : 0, before = block_excl_scan32<kThreads>(v, s_w, total);
    if (t < kGroups) s_g[t] = before;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint32_t p = j * kThreads + t;
    if (p < cnt) {
      const uint32_t run = s_g[p >> 6] + br[j];
      s_up[p] = (uint16_t)run;
      if ((flags >> j) & 1) s_col[run] = col[j];
    }
  }
  if (t == 0) {
    s_up[cnt] = (uint16_t)total;
    sub_unique[sub] = total;
  }
  __syncthreads();
  uint32_t* const out = reinterpret_cast<uint32_t*>(x + off);
  for (uint32_t p = t; p < total; p += kThreads) out[p] = s_col[p];
  for (int64_t r = row0 + t; r < rows; r += kThreads) {
    const uint64_t p0 = P[r], p1 = P[r + 1];
    if (p0 >= pos_end) break;
    const uint32_t i0 = (uint32_t)((p0 > pos ? p0 : pos) - pos), i1 = (uint32_t)((p1 < pos_end ? p1 : pos_end) - pos);
    const uint32_t u = s_up[s_start[i1]] - s_up[s_start[i0]];
    if (p0 >= pos && p1 <= pos_end) row_unique[r] = u;
    else if (u) atomicAdd(&row_unique[r], u);
  }
}

// The unique columns of every sub-bucket to their place in cols.
__global__ void __launch_bounds__(kBlock) k_compact(const uint64_t* __restrict__ x,
                                                    const uint64_t* __restrict__ sub_off,
                                                    const uint32_t* __restrict__ sub_unique,
                                                    const uint64_t* __restrict__ out_off,
                                                    const unsigned long long* __restrict__ info,
                                                    uint32_t* __restrict__ cols) {
  const uint32_t sub = blockIdx.x;
  if (sub >= info[I_SUBS]) return;
  const uint32_t n = sub_unique[sub];
  const uint32_t* const src = reinterpret_cast<const uint32_t*>(x + sub_off[sub]);
  uint32_t* const dst = cols + out_off[sub];
  for (uint32_t p = threadIdx.x; p < n; p += kBlock) dst[p] = src[p];
}

// Entries (position in the L1 bucket, column) back to (row, column) keys, for
// the radix sort: the row is the last one with P[row] <= position.
__global__ void __launch_bounds__(kBlock) k_entry_keys(const uint64_t* __restrict__ in, uint64_t n,
                                                       const uint64_t* __restrict__ P, int64_t rows,
                                                       const uint64_t* __restrict__ base, int nb1,
                                                       uint64_t* __restrict__ keys) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock) {
    int a = 0, z = nb1 - 1;  // the entry's bucket: the last one that starts at or before it
    while (a < z) {
      const int mid = (a + z + 1) >> 1;
      if (base[mid] <= i) a = mid; else z = mid - 1;
    }
    const uint64_t e = in[i], p = base[a] + (e >> 32);
    int64_t lo = 0, hi = rows - 1;
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) >> 1;
      if (P[mid] <= p) lo = mid; else hi = mid - 1;
    }
    keys[i] = ((uint64_t)lo << 32) | (uint32_t)e;
  }
}

}  // namespace g5
