// g5_msbfs.hip -- batched multi-source BFS: up to 64 roots share one sweep.
//
// Lane r of every 64-bit word belongs to root r.  Per vertex (degree-ordered
// new ids, rows [0, n_rows)):
//   seen[v]        lanes that have reached v
//   fr[l][v]       lanes for which v is at level l (the frontier of level l+1);
//                  kept for every level, so the per-root level arrays are
//                  rebuilt after the run without any extra store in the sweep
// Each level is a push or a pull step, chosen from the edge count of the
// frontier union (the direction-optimizing rule applied to the union):
//   push  the union's rows form a chunked virtual edge list (as in the
//         single-root top-down); target w receives front[u] with one
//         64-bit atomicOr, filtered by a plain load of next[w]; k_ms_finish
//         then masks the lanes new to w and folds them into seen
//   pull  one lane per vertex: the lanes it still lacks (and whose frontier
//         is not empty) are collected by OR-ing the neighbours' frontier
//         words in ascending (highest degree first) order until every needed
//         lane is found or the row ends, rows over 8 entries by groups of 16
//         lanes.  On request a 1-bit-per-vertex "frontier word is not zero"
//         bitmap (n/8 bytes) is tested before an 8-byte frontier word
// Small graphs are bound by launches: a level is at most five (select, ready,
// push, pull, publish), a pull two, a start two (S12, 64 roots: 41 launches
// and 242 us, now 24 and 162).
// Per-lane levels equal the single-root BFS levels of the same root.
#include "g5_answers.hpp"
#include "g5_ctx.hpp"
#include "g5_frontier.hpp"
#include "g5_ms_device.hpp"

#include <algorithm>
#include <cstring>

namespace g5 {

constexpr int kMsCounters = kMsLanes + 128;  // level counters, a list count, per-lane counts and degree sums
constexpr size_t kMsCounterWords = (size_t)kMsStripes * kMsStride;
static_assert(kMsCounters <= kMsStride, "a counter copy holds every counter");

// Device clock at the start of a batch and of a level (m.stamps); a level's
// first kernel stamps it, and every publish sends the times since both.
// (Events around each level took 7 us a level of the stream's time.)
enum { T_BATCH = 0, T_LEVEL = 1, T_NUM = 2 };
__device__ __forceinline__ void ms_stamp(uint64_t* stamp) {
  if (stamp && blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
}
__global__ void k_ms_stamp(uint64_t* stamp) { ms_stamp(stamp); }

__global__ void __launch_bounds__(kBlock) k_ms_clear(uint64_t* __restrict__ a, uint64_t* __restrict__ b,
                                                     int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    a[i] = 0;
    b[i] = 0;
  }
}

// Marks every active root in seen and fr0 and counts the level-0 union: one
// wave, lane r takes root r; of the roots sharing a vertex, the lane whose
// atomic OR finds its word still zero counts the vertex.
__global__ void k_ms_roots(const uint32_t* __restrict__ old2new, const int64_t* __restrict__ roots, int nroots,
                           int64_t rows, const uint64_t* __restrict__ offsets, uint64_t* __restrict__ seen,
                           uint64_t* __restrict__ fr0, unsigned long long* __restrict__ c) {
  if (blockIdx.x != 0 || threadIdx.x >= 64) return;
  const int r = threadIdx.x;
  bool act = false, first = false;
  uint64_t deg = 0;
  if (r < nroots && roots[r] >= 0) {  // unused lanes hold -1
    const uint32_t v = old2new[roots[r]];
    act = (int64_t)v < rows;  // a root without edges discovers nothing
    if (act) {
      const unsigned long long bit = 1ull << r;
      atomicOr((unsigned long long*)(seen + v), bit);
      first = atomicOr((unsigned long long*)(fr0 + v), bit) == 0;
      if (first) deg = offsets[v + 1] - offsets[v];
    }
  }
  const uint64_t live = __ballot(act);
  const uint64_t nz = (uint64_t)__popcll(__ballot(first));
  const uint64_t fdeg = wave_sum(deg);
  if (r == 0) {
    c[M_LIVE] = live;
    c[M_PAIRS] = 0;
    c[M_NZ] = nz;
    c[M_FDEG] = fdeg;
  }
}

// The roots of a level-by-level batch, in the argument block.
struct MsRoots {
  int64_t root[64];
  int n;
};

// A batch's start in two launches.  k_ms_begin clears the reached lanes, level
// 0's frontier words (the ones its last run marked, or all), their marks and
// the level counters (which every publish clears again); k_ms_place puts the
// roots in and publishes the first level's counters.
__global__ void __launch_bounds__(kBlock) k_ms_begin(uint64_t* __restrict__ seen, uint64_t* __restrict__ fr0,
                                                     uint64_t* __restrict__ nz0, int64_t rows, int64_t words,
                                                     int marked, unsigned long long* __restrict__ counters,
                                                     uint64_t* __restrict__ stamps) {
  ms_stamp(stamps + T_BATCH);
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x, stride = (int64_t)gridDim.x * kBlock;
  for (int64_t v = t; v < rows; v += stride) {
    seen[v] = 0;
    if (!marked) fr0[v] = 0;
  }
  for (int64_t wd = t; wd < words; wd += stride) {
    if (marked)
      for (uint64_t b = nz0[wd]; b; b &= b - 1) {
        const int64_t v = wd * 64 + __builtin_ctzll(b);
        if (v < rows) fr0[v] = 0;
      }
    nz0[wd] = 0;
  }
  for (int64_t i = t; i < (int64_t)kMsCounterWords; i += stride) counters[i] = 0;
}

__global__ void __launch_bounds__(64) k_ms_place(const uint32_t* __restrict__ old2new, MsRoots roots, int64_t rows,
                                                 const uint64_t* __restrict__ offsets, uint64_t* __restrict__ seen,
                                                 uint64_t* __restrict__ fr0, uint64_t* __restrict__ nz0,
                                                 Published* __restrict__ pub, uint64_t seq,
                                                 const uint64_t* __restrict__ stamps) {
  const int r = threadIdx.x;
  bool act = false, first = false;
  uint64_t deg = 0;
  if (r < roots.n) {
    const uint32_t v = old2new[roots.root[r]];
    act = (int64_t)v < rows;  // a root without edges discovers nothing
    if (act) {
      const unsigned long long bit = 1ull << r;
      atomicOr((unsigned long long*)(seen + v), bit);
      atomicOr((unsigned long long*)(nz0 + (v >> 6)), 1ull << (v & 63));
      first = atomicOr((unsigned long long*)(fr0 + v), bit) == 0;
      if (first) deg = offsets[v + 1] - offsets[v];
    }
  }
  const uint64_t live = __ballot(act);
  const uint64_t nz = (uint64_t)__popcll(__ballot(first));
  const uint64_t fdeg = wave_sum(deg);
  if (r < T_NUM) publish(pub + kMsCounters + r, wall_clock64() - stamps[T_BATCH], seq);
  if (r < M_NUM) publish(pub + r, r == M_LIVE ? live : r == M_NZ ? nz : r == M_FDEG ? fdeg : 0, seq);
}

// Level-0 nonzero bitmap: the root vertices (lane r, root r).
__global__ void k_ms_roots_nz(const uint32_t* __restrict__ old2new, const int64_t* __restrict__ roots, int nroots,
                              int64_t rows, uint64_t* __restrict__ nz0) {
  const int r = threadIdx.x;
  if (blockIdx.x != 0 || r >= nroots || roots[r] < 0) return;
  const uint32_t v = old2new[roots[r]];
  if ((int64_t)v < rows) atomicOr((unsigned long long*)(nz0 + (v >> 6)), 1ull << (v & 63));
}

__global__ void __launch_bounds__(kBlock) k_ms_push(const uint32_t* __restrict__ queue, int64_t nf,
                                                    const uint64_t* __restrict__ prefix,
                                                    const uint32_t* __restrict__ chunk_rows,
                                                    const uint64_t* __restrict__ offsets,
                                                    const uint32_t* __restrict__ cols,
                                                    const uint64_t* __restrict__ front, uint64_t* next,
                                                    uint64_t lanes) {
  // front[u] (its lanes in `lanes`) goes to every target; lanes the target
  // has seen are dropped when k_ms_finish (or the merging pull) folds next
  // into seen.  prefix[nf] is the edge count: nf may be an upper bound whose
  // tail entries have degree 0.
  __shared__ ChunkRows cr;
  const uint64_t E = prefix[nf];
  for (uint64_t chunk = blockIdx.x; chunk * kEpb < E; chunk += gridDim.x) {
    const uint64_t e0 = chunk * kEpb;
    const uint64_t e1 = (e0 + kEpb < E) ? e0 + kEpb : E;
    const int cnt = stage_chunk(chunk, chunk_rows, queue, prefix, offsets, cr);
    walk_strided(e0, e1, cnt, cr, cols, [&](uint32_t w, uint32_t u) {
      const uint64_t m = front[u] & lanes;
      if (m & ~__atomic_load_n(next + w, __ATOMIC_RELAXED))
        atomicOr((unsigned long long*)(next + w), (unsigned long long)m);
    });
    __syncthreads();
  }
}

// k_ms_push that also lists the vertices it touches: the one atomicOr that
// finds a target's word still zero (next was cleared for the level) appends
// the target, staged in LDS and appended with one global atomic per chunk.
__global__ void __launch_bounds__(kBlock) k_ms_push_touch(const uint32_t* __restrict__ queue, int64_t nf,
                                                          const uint64_t* __restrict__ prefix,
                                                          const uint32_t* __restrict__ chunk_rows,
                                                          const uint64_t* __restrict__ offsets,
                                                          const uint32_t* __restrict__ cols,
                                                          const uint64_t* __restrict__ front, uint64_t* next,
                                                          uint32_t* __restrict__ list,
                                                          unsigned long long* __restrict__ list_count) {
  __shared__ ChunkRows cr;
  __shared__ uint32_t s_q[kEpb];
  __shared__ uint32_t s_qn;
  __shared__ uint64_t s_qbase;
  const uint64_t E = prefix[nf];
  for (uint64_t chunk = blockIdx.x; chunk * kEpb < E; chunk += gridDim.x) {
    const uint64_t e0 = chunk * kEpb;
    const uint64_t e1 = (e0 + kEpb < E) ? e0 + kEpb : E;
    if (threadIdx.x == 0) s_qn = 0;
    const int cnt = stage_chunk(chunk, chunk_rows, queue, prefix, offsets, cr);
    walk_strided(e0, e1, cnt, cr, cols, [&](uint32_t w, uint32_t u) {
      const uint64_t m = front[u];
      if (m & ~__atomic_load_n(next + w, __ATOMIC_RELAXED)) {
        const uint64_t old = atomicOr((unsigned long long*)(next + w), (unsigned long long)m);
        if (old == 0) s_q[atomicAdd(&s_qn, 1u)] = w;
      }
    });
    __syncthreads();
    if (threadIdx.x == 0) s_qbase = s_qn ? atomicAdd(list_count, (unsigned long long)s_qn) : 0;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < s_qn; j += kBlock) list[s_qbase + j] = s_q[j];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kBlock) k_ms_finish_list(uint64_t* __restrict__ seen, uint64_t* __restrict__ next,
                                                           uint64_t* __restrict__ nz_next,
                                                           const uint64_t* __restrict__ offsets,
                                                           const uint32_t* __restrict__ list,
                                                           const unsigned long long* __restrict__ list_count,
                                                           unsigned long long* __restrict__ c, LaneEpi epi_in,
                                                           int lane_stats) {
  const uint64_t n = *list_count;
  if (lane_stats) {
    LaneEpi epi = epi_in;  // a copy in registers: the epilogue accumulates per thread
    epi.lane_nq = ms_stripe(epi.lane_nq);
    ms_finish_list_body(seen, next, nz_next, offsets, list, n, ms_stripe(c), blockIdx.x, gridDim.x, epi);
  } else {
    ms_finish_list_body(seen, next, nz_next, offsets, list, n, ms_stripe(c), blockIdx.x, gridDim.x);
  }
}

__global__ void __launch_bounds__(kBlock) k_ms_finish(uint64_t* __restrict__ seen, uint64_t* __restrict__ next,
                                                      uint64_t* __restrict__ nz_next,
                                                      const uint64_t* __restrict__ offsets, int64_t rows,
                                                      unsigned long long* __restrict__ c) {
  ms_finish_body(seen, next, nz_next, offsets, rows, ms_stripe(c), blockIdx.x, gridDim.x);
}

template <int kU, int kW, int kRows = 64>
__global__ void __launch_bounds__(kBlock) k_ms_pull(uint64_t* __restrict__ seen, const uint64_t* __restrict__ front,
                                                    const uint64_t* __restrict__ nz_front, uint64_t* __restrict__ next,
                                                    uint64_t* __restrict__ nz_next,
                                                    const uint32_t* __restrict__ first_nbr,
                                                    const uint64_t* __restrict__ offsets,
                                                    const uint32_t* __restrict__ cols, int64_t rows,
                                                    uint64_t live_in, int mode, const uint64_t* __restrict__ pack,
                                                    const uint64_t* __restrict__ compact, uint32_t filter_from,
                                                    unsigned long long* __restrict__ c, uint64_t* __restrict__ miss,
                                                    uint64_t* __restrict__ stamp) {
  ms_stamp(stamp);
  const FrontView fv{front, nz_front, pack, compact, mode, filter_from};
  ms_pull_body<NoEpilogue, kU, kW, kRows>(seen, fv, next, nz_next, first_nbr, offsets, cols, rows, live_in, ms_stripe(c),
                                   blockIdx.x, gridDim.x, ~UINT64_C(0), NoEpilogue(), false, miss);
}

// The pull of a tail level over the listed vertices (see ms_pull_list_body).
__global__ void __launch_bounds__(kBlock) k_ms_pull_list(uint64_t* __restrict__ seen, const uint64_t* __restrict__ front,
                                                         uint64_t* __restrict__ next, uint64_t* __restrict__ nz_next,
                                                         const uint32_t* __restrict__ first_nbr,
                                                         const uint64_t* __restrict__ offsets,
                                                         const uint32_t* __restrict__ cols,
                                                         const uint32_t* __restrict__ list,
                                                         const uint64_t* __restrict__ list_count, uint64_t live_in,
                                                         uint64_t* __restrict__ miss,
                                                         unsigned long long* __restrict__ c) {
  const FrontView fv{front, nullptr, nullptr, nullptr, kFrontPlain, 0};
  ms_pull_list_body(seen, fv, next, nz_next, first_nbr, offsets, cols, list, *list_count, live_in, miss,
                    ms_stripe(c), blockIdx.x, gridDim.x);
}

// --- per-root directions (lane_rule 1) ---
__global__ void __launch_bounds__(kBlock) k_ms_finish_lanes(uint64_t* __restrict__ seen, uint64_t* __restrict__ next,
                                                            uint64_t* __restrict__ nz_next,
                                                            const uint64_t* __restrict__ offsets, int64_t rows,
                                                            unsigned long long* __restrict__ c, LaneEpi epi_in) {
  LaneEpi epi = epi_in;  // a copy in registers: the epilogue accumulates per thread
  epi.lane_nq = ms_stripe(epi.lane_nq);
  ms_finish_body(seen, next, nz_next, offsets, rows, ms_stripe(c), blockIdx.x, gridDim.x, ~UINT64_C(0), epi);
}

// Pull for the lanes in live_in; with merge, next already holds this level's
// pushed lanes, which are folded in.
template <int kU, int kW, int kRows = 64>
__global__ void __launch_bounds__(kBlock) k_ms_pull_lanes(uint64_t* __restrict__ seen, const uint64_t* __restrict__ front,
                                                          const uint64_t* __restrict__ nz_front, uint64_t* __restrict__ next,
                                                          uint64_t* __restrict__ nz_next,
                                                          const uint32_t* __restrict__ first_nbr,
                                                          const uint64_t* __restrict__ offsets,
                                                          const uint32_t* __restrict__ cols, int64_t rows,
                                                          uint64_t live_in, int filter, int merge,
                                                          unsigned long long* __restrict__ c, LaneEpi epi_in) {
  LaneEpi epi = epi_in;  // a copy in registers: the epilogue accumulates per thread
  epi.lane_nq = ms_stripe(epi.lane_nq);
  const FrontView fv{front, nz_front, nullptr, nullptr, filter ? kFrontFilter : kFrontPlain, 0};
  ms_pull_body<LaneEpi, kU, kW, kRows>(seen, fv, next, nz_next, first_nbr, offsets, cols, rows, live_in, ms_stripe(c),
                                blockIdx.x, gridDim.x, ~UINT64_C(0), epi, merge != 0);
}

// One bit per vertex whose frontier word has one of `lanes`.
__global__ void __launch_bounds__(kBlock) k_ms_select(const uint64_t* __restrict__ front, int64_t rows, uint64_t lanes,
                                                      uint64_t* __restrict__ nz_sel, uint64_t* __restrict__ stamp) {
  ms_stamp(stamp);
  ms_select_body(front, rows, lanes, nz_sel, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(kBlock) k_ms_collect(const uint32_t* __restrict__ chunk_rows, uint64_t nchunks,
                                                       const uint64_t* __restrict__ nz_sel, uint32_t* __restrict__ list,
                                                       unsigned* count) {
  ms_collect_chunks_body(chunk_rows, nchunks, nz_sel, list, count, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(kBlock) k_ms_push_list(const uint32_t* __restrict__ list, const unsigned* count,
                                                         const uint32_t* __restrict__ chunk_rows, uint64_t nnz,
                                                         const uint64_t* __restrict__ offsets,
                                                         const uint32_t* __restrict__ cols,
                                                         const uint64_t* __restrict__ front,
                                                         const uint64_t* __restrict__ nz_sel, uint64_t* next,
                                                         uint64_t lanes) {
  __shared__ SweepLds L;
  ms_push_list_body(list, count, chunk_rows, nnz, offsets, cols, front, nz_sel, next, L, blockIdx.x, gridDim.x, lanes);
}

__global__ void __launch_bounds__(kBlock) k_ms_sweep_clear(const uint32_t* __restrict__ chunk_rows,
                                                           uint64_t nchunks, const uint64_t* __restrict__ offsets,
                                                           uint64_t* __restrict__ next) {
  ms_sweep_clear_body(chunk_rows, nchunks, offsets, next, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(kBlock) k_ms_sweep(const uint32_t* __restrict__ chunk_rows, uint64_t nnz,
                                                     const uint64_t* __restrict__ offsets,
                                                     const uint32_t* __restrict__ cols,
                                                     const uint64_t* __restrict__ front,
                                                     const uint64_t* __restrict__ nz_front,
                                                     uint64_t* __restrict__ next) {
  __shared__ SweepLds L;
  ms_sweep_body(chunk_rows, nnz, offsets, cols, front, nz_front, next, L, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// Persistent level-fused batch: one launch runs every level, the grid meeting
// at a barrier between the phases of a level.  All blocks read the same level
// counters after a barrier and so take the same direction decision; the loop
// ends when no lane discovers anything, when the preallocated frontier-word
// arrays run out (the host loop continues from there), or when a barrier wait
// exceeds its deadline (then every block leaves and the host reports it).
// ---------------------------------------------------------------------------
// Two-level arrival: workgroups count in on one of up to kBarMaxGroups group
// counters (kBarGroup each, one 128-byte line apiece), the last of a group
// counts in on the top counter, and the last group flips the generation that
// everyone waits on; this keeps the atomics on any one address to a few tens
// per barrier instead of one per workgroup.
// Tail pull levels go list-driven once fewer than rows / kListBelow (root,
// vertex) pairs are unreached.
constexpr double kListBelow = 16.0;

// The listed pulls run on at most this many workgroups: their list is far
// shorter than its bound, and workgroups that find nothing to do still cost
// (SCALE 28, per listed level: 0.070 ms on up to 4,096, 0.093 on 16,384).
constexpr int64_t kListGrid = 2048;

// Pulls of graphs up to this many words take 16 rows a turn instead of 64: a
// wave with the 64 rows of the largest hubs outlasts the rest of a small
// graph (the first pull of S12 87 us, now 49; S16 120, 68; S18 152, 95).  A
// pull that follows finds most rows done, and turns cost more than they give
// from S19 on (5,200 words: 9 us a level, now 20); a first one loses from S21
// (167 us, 178; S20 133, 113).
constexpr int64_t kPartWords = 4096;
constexpr int64_t kPartWordsFirst = 12288;

// Below this many entries a root waits for the union one level only (lane_rule
// 1): a level costs its launches there, two for a pull and four for a push,
// and long graphs never have a union large enough (2 and 8 roots, us, waiting
// and not: a path of 200 6,214 / 6,047 and 3,467 / 4,254, 128 x 1,024 vertices
// in a grid with chords 3,998 / 7,038 and 2,834 / 3,771).  The one level stays
// for graphs that grow: from the next on their union is large enough, and a
// mixed level in between costs S14 to S18 5 to 8 %.
constexpr int64_t kUnionFrom = INT64_C(1) << 22;

// A push level lists the vertices it touches when its frontier edges times
// this are fewer than the rows (the touched vertices are at most the edges).
constexpr double kTouchBelow = 8.0;

constexpr unsigned kBarGroup = 16;
constexpr unsigned kBarMaxGroups = 1024;
struct GridBarrier {
  unsigned count;
  unsigned gen;
  unsigned abort;
  unsigned pad[29];
  unsigned group[kBarMaxGroups][32];
};

// Returns false (in every thread of the block) once any block has given up.
__device__ __forceinline__ bool grid_barrier(GridBarrier* b, unsigned nblk, long long deadline) {
  __shared__ int s_ok;
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = 1;
    const unsigned g = __hip_atomic_load(&b->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence();
    const unsigned grp = blockIdx.x / kBarGroup;
    const unsigned ngroups = (nblk + kBarGroup - 1) / kBarGroup;
    const unsigned gsize = (grp + 1 < ngroups) ? kBarGroup : nblk - grp * kBarGroup;
    bool last = false;
    if (__hip_atomic_fetch_add(&b->group[grp][0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gsize - 1) {
      __hip_atomic_store(&b->group[grp][0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = __hip_atomic_fetch_add(&b->count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == ngroups - 1;
    }
    if (last) {
      __hip_atomic_store(&b->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_add(&b->gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      // relaxed polls (an acquire per poll would invalidate the caches the
      // still-working workgroups depend on); one acquire fence after
      while (__hip_atomic_load(&b->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g) {
        if (__hip_atomic_load(&b->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
            wall_clock64() > deadline) {
          __hip_atomic_store(&b->abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ok = 0;
          break;
        }
        __builtin_amdgcn_s_sleep(8);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (__hip_atomic_load(&b->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ok = 0;
    s_ok = ok;
  }
  __syncthreads();
  return s_ok != 0;
}

struct MsPersistArgs {
  const uint64_t* offsets;
  const uint32_t* cols;
  const uint32_t* first_nbr;
  const uint32_t* sweep_rows;  // first/last row per sweep chunk
  int64_t rows;
  uint64_t nnz;
  uint64_t sweep_chunks;
  uint64_t* seen;
  uint64_t* const* fr;          // frontier words of levels 0 .. max_levels-1
  uint64_t* nz0;
  uint64_t* nz1;
  unsigned long long* cnt;      // [max_levels][M_NUM]; level 0 filled by k_ms_roots, rest zero
  long long* ts;                // [max_levels] wall clock at the end of each level
  int* dir;                     // [max_levels] level kind (1 push, 0 pull, 2 sweep)
  int* done_levels;             // last level completed
  GridBarrier* bar;
  uint32_t* chunk_list;         // sweep chunks holding a frontier row (push levels)
  unsigned* chunk_count;
  double push_limit;            // nnz / alpha
  double sweep_below;           // sweep while reached pairs < sweep_below x roots x rows
  int pull_filter;              // pull reads a frontier word only after its nonzero bit
  double pull_unseen_frac;      // pull whenever fewer than this fraction of pairs are unreached
  int max_levels;
  long long timeout_ticks;      // per-barrier wait bound (wall clock ticks)
};

// kWaves: waves per SIMD the compiler must fit (register budget 512 / kWaves).
template <int kWaves>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kWaves, kWaves)))
k_ms_persistent(MsPersistArgs a) {
  __shared__ SweepLds L;
  const unsigned bid = blockIdx.x, nblk = gridDim.x;
  const int64_t words = (a.rows + 63) / 64;
  if (bid == 0 && threadIdx.x == 0) a.ts[0] = wall_clock64();
  uint64_t live = __hip_atomic_load(&a.cnt[M_LIVE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const double roots_live = (double)__popcll(live);
  const double sweep_limit = a.sweep_below * roots_live * (double)a.rows;
  const double total_pairs = roots_live * (double)a.rows;
  double reached = roots_live;
  int l = 0;
  while (live && l + 1 < a.max_levels) {
    const unsigned long long* cp = a.cnt + (size_t)l * M_NUM;
    const uint64_t fdeg = __hip_atomic_load(&cp[M_FDEG], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    ++l;
    unsigned long long* c = a.cnt + (size_t)l * M_NUM;
    const uint64_t* front = a.fr[l - 1];
    uint64_t* next = a.fr[l];
    const uint64_t* nz_front = ((l - 1) & 1) ? a.nz1 : a.nz0;
    uint64_t* nz_next = (l & 1) ? a.nz1 : a.nz0;
    // push a small frontier union, unless nearly every pair is reached (then
    // a pull touches little beyond the seen words)
    const bool push = (double)fdeg < a.push_limit && total_pairs - reached >= a.pull_unseen_frac * total_pairs;
    const bool sweep = !push && a.sweep_chunks && reached < sweep_limit;
    const long long deadline = wall_clock64() + a.timeout_ticks;
    if (push) {
      ms_zero_body(next, a.rows, bid, nblk);
      if (bid == 0 && threadIdx.x == 0) *a.chunk_count = 0;
      if (!grid_barrier(a.bar, nblk, deadline)) return;
      ms_collect_chunks_body(a.sweep_rows, a.sweep_chunks, nz_front, a.chunk_list, a.chunk_count, bid, nblk);
      if (!grid_barrier(a.bar, nblk, deadline)) return;
      ms_push_list_body(a.chunk_list, a.chunk_count, a.sweep_rows, a.nnz, a.offsets, a.cols, front, nz_front,
                        next, L, bid, nblk);
      if (!grid_barrier(a.bar, nblk, deadline)) return;
      ms_finish_body(a.seen, next, nz_next, a.offsets, a.rows, c, bid, nblk);
    } else if (sweep) {
      ms_sweep_clear_body(a.sweep_rows, a.sweep_chunks, a.offsets, next, bid, nblk);
      if (!grid_barrier(a.bar, nblk, deadline)) return;
      ms_sweep_body(a.sweep_rows, a.nnz, a.offsets, a.cols, front, nz_front, next, L, bid, nblk);
      if (!grid_barrier(a.bar, nblk, deadline)) return;
      ms_finish_body(a.seen, next, nz_next, a.offsets, a.rows, c, bid, nblk);
    } else {
      const FrontView fv{front, nz_front, nullptr, nullptr, a.pull_filter == 1 ? kFrontFilter : kFrontPlain, 0};
      ms_pull_body(a.seen, fv, next, nz_next, a.first_nbr, a.offsets, a.cols, a.rows, live, c, bid, nblk);
    }
    if (!grid_barrier(a.bar, nblk, deadline)) return;
    live = __hip_atomic_load(&c[M_LIVE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    reached += (double)__hip_atomic_load(&c[M_PAIRS], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (bid == 0 && threadIdx.x == 0) {
      a.ts[l] = wall_clock64();
      a.dir[l] = push ? 1 : (sweep ? 2 : 0);
      *a.done_levels = l;
    }
  }
  (void)words;
}

// Zero fill (graph-capturable, unlike a memset node).
__global__ void __launch_bounds__(kBlock) k_ms_fill(uint64_t* __restrict__ a, int64_t n) {
  ms_zero_body(a, n, blockIdx.x, gridDim.x);
}

// A lane's level is the first level whose frontier word holds it.  The levels'
// frontier words and nonzero bitmaps travel in the argument block.
constexpr int kMsArgLevels = 24;
struct LevelWords {
  const uint64_t* fr[kMsArgLevels];
  const uint64_t* nz[kMsArgLevels];  // null where a level's bitmap does not describe its words
  const uint64_t* const* more;       // the frontier words again, for deeper searches
  int n;
  __device__ const uint64_t* words(int i) const { return i < kMsArgLevels ? fr[i] : more[i]; }
};

// Levels by original id: 4 consecutive ids per thread, their words of one
// level in flight together.  For graphs whose frontier words sit in the L2s.
__global__ void __launch_bounds__(kBlock) k_ms_levels(const uint32_t* __restrict__ old2new, int64_t n, int64_t rows,
                                                      LevelWords lw, int lane, int64_t root,
                                                      uint8_t* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q * 4 < n; q += stride) {
    const int m = n < 4 ? (int)n : 4;  // n is a power of two
    uint32_t nv[4];
    uint32_t l[4];
    bool open[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      nv[j] = j < m ? old2new[q * 4 + j] : 0xFFFFFFFFu;
      l[j] = 0xFF;
      open[j] = (int64_t)nv[j] < rows;
    }
    for (int i = 0; i < lw.n && (open[0] || open[1] || open[2] || open[3]); ++i) {
      const uint64_t* f = lw.words(i);
      uint64_t x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = open[j] ? f[nv[j]] : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((x[j] >> lane) & 1) {
          l[j] = i;
          open[j] = false;
        }
    }
    const int64_t r = root - q * 4;
    if (r >= 0 && r < 4) {  // also a root without edges, which is no row of the CSR
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (r == j) l[j] = 0;
    }
    if (m == 4) {
      reinterpret_cast<uint32_t*>(out)[q] = l[0] | (l[1] << 8) | (l[2] << 16) | (l[3] << 24);
    } else {
      for (int j = 0; j < m; ++j) out[j] = (uint8_t)l[j];
    }
  }
}

// Levels by row, for larger graphs: a lane takes 4 consecutive rows and reads
// a level's words of them only where the level's bitmap has one that is still
// open, the bitmap words of 4 levels in flight together; the lookup by
// original id is then one byte each (k_make_levels) instead of a word per
// level.  A lane's levels of S26 (34 M rows, 0.4 GB read), one row per thread
// and a bitmap word at a time: 390 us, bound by the chain of loads.
__global__ void __launch_bounds__(kBlock) k_ms_row_levels(LevelWords lw, int64_t rows, int lane_bit,
                                                          uint8_t* __restrict__ out) {
  const int64_t quads = (rows + 3) / 4, stride = (int64_t)gridDim.x * kBlock;
  for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q < quads; q += stride) {
    const int64_t v = q * 4;
    const int m = rows - v < 4 ? (int)(rows - v) : 4;
    const int sh = (int)(v & 63);
    uint32_t open = (1u << m) - 1, l = 0xFFFFFFFFu;
    for (int i0 = 0; i0 < lw.n && open; i0 += 4) {
      uint32_t nz[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = i0 + j;
        const uint64_t* w = i < lw.n && i < kMsArgLevels ? lw.nz[i] : nullptr;
        nz[j] = i >= lw.n ? 0u : w ? (uint32_t)(w[v >> 6] >> sh) & 15u : 15u;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (!(nz[j] & open)) continue;
        const uint64_t* f = lw.words(i0 + j) + v;
        alignas(16) uint64_t x[4];
        if (m == 4) {
          *reinterpret_cast<ulonglong2*>(x) = *reinterpret_cast<const ulonglong2*>(f);
          *reinterpret_cast<ulonglong2*>(x + 2) = *reinterpret_cast<const ulonglong2*>(f + 2);
        } else {
          for (int k = 0; k < 4; ++k) x[k] = k < m ? f[k] : 0;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (((open >> k) & 1) && ((x[k] >> lane_bit) & 1)) {
            l = (l & ~(0xFFu << (8 * k))) | (uint32_t)(i0 + j) << (8 * k);
            open &= ~(1u << k);
          }
      }
    }
    if (m == 4) {
      reinterpret_cast<uint32_t*>(out)[q] = l;
    } else {
      for (int k = 0; k < m; ++k) out[v + k] = (uint8_t)(l >> (8 * k));
    }
  }
}

// Traversed-edge numerators of all lanes: sum of weight over the vertices
// each lane reached.  Vertices reached by every lane go to one sum; for the
// others, thread i of a wave sums lane i's weights (readlane walk).  Workgroups
// add to one of kTepsStripes copies; k_ms_teps_publish sums and clears them.
// Bound by the words and weights read (12 B per row); one copy of the sums
// held the workgroups up at its words (12 ns an add: S22 82 us, now 29).
constexpr int kTepsStripes = 16;
constexpr int kTepsStride = 72;
__global__ void __launch_bounds__(kBlock) k_ms_teps(const uint64_t* __restrict__ seen,
                                                    const uint32_t* __restrict__ weight, int64_t rows,
                                                    uint64_t all, unsigned long long* __restrict__ acc) {
  __shared__ unsigned long long s_acc[65];
  if (threadIdx.x < 65) s_acc[threadIdx.x] = 0;
  __syncthreads();
  const int me = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (kBlock / 64);
  uint64_t full = 0, mine = 0;
  for (int64_t wd = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); wd * 64 < rows; wd += nwaves) {
    const int64_t v = wd * 64 + me;
    const uint64_t x = v < rows ? seen[v] : 0;
    const uint32_t w = v < rows ? weight[v] : 0;
    if (x == all) full += w;
    uint64_t m = __ballot(x != 0 && x != all);
    while (m) {
      const int t = __builtin_ctzll(m);
      m &= m - 1;
      const uint32_t xlo = __builtin_amdgcn_readlane((uint32_t)x, t);
      const uint32_t xhi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), t);
      const uint32_t wt = __builtin_amdgcn_readlane(w, t);
      mine += ((me < 32 ? xlo >> me : xhi >> (me - 32)) & 1) ? wt : 0;
    }
  }
  full = wave_sum(full);
  if (me == 0 && full) atomicAdd(&s_acc[64], (unsigned long long)full);
  if (mine) atomicAdd(&s_acc[me], (unsigned long long)mine);
  __syncthreads();
  if (threadIdx.x < 65 && s_acc[threadIdx.x])
    atomicAdd(acc + (blockIdx.x % kTepsStripes) * kTepsStride + threadIdx.x, s_acc[threadIdx.x]);
}

__global__ void __launch_bounds__(128) k_ms_teps_publish(unsigned long long* __restrict__ acc, Published* pub,
                                                         uint64_t seq) {
  const int t = threadIdx.x;
  if (t > 64) return;
  uint64_t sum = 0;
#pragma unroll
  for (int i = 0; i < kTepsStripes; ++i) {
    sum += acc[i * kTepsStride + t];
    acc[i * kTepsStride + t] = 0;
  }
  publish(pub + t, sum, seq);
}

// --- batched byte model (evaluated after the run from the per-level words) ---
// level l: 24 n + sum over vertices with a needed pulled lane of (8 + 12 k),
// k = probes until every needed lane is found (the row length if not), +
// sum over vertices whose frontier word holds a pushed lane of (8 + 12 deg):
// the word, then per entry the column and the target's next word.  With one
// direction for all roots every level is costed as a pull of all lanes.
__global__ void __launch_bounds__(kBlock) k_ms_model(const uint64_t* const* __restrict__ fr, int l,
                                                     uint64_t lanes, uint64_t push_lanes,
                                                     const uint64_t* __restrict__ offsets,
                                                     const uint32_t* __restrict__ cols, int64_t rows,
                                                     unsigned long long* __restrict__ acc) {
  uint64_t b = 0;
  for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < rows; v += (int64_t)gridDim.x * kBlock) {
    uint64_t seen_before = 0;
    for (int i = 0; i < l; ++i) seen_before |= fr[i][v];
    const uint64_t need = ~seen_before & lanes;
    const uint64_t s = offsets[v], e = offsets[v + 1];
    if (fr[l - 1][v] & push_lanes) b += 8 + 12 * (e - s);
    if (!need || s == e) continue;
    uint64_t a = 0, k = 0;
    for (uint64_t j = s; j < e; ++j) {
      ++k;
      a |= fr[l - 1][cols[j]];
      if ((a & need) == need) break;
    }
    b += 8 + 12 * k;
  }
  block_add(b, acc);
}

// ---------------------------------------------------------------------------
// Host
// ---------------------------------------------------------------------------
// Frontier levels preallocated by g5_batch_prepare (a SCALE 28 batch takes 9).
constexpr int kMsPreLevels = 16;

// The compact frontier copy of the pull (compact_below > 0).
void ms_alloc_compact(g5_ctx* ctx) {
  MsState& m = ctx->ms;
  const int64_t rows = ctx->graph.n_rows;
  m.pack.alloc(2 * ((rows + 63) / 64));
  m.compact.alloc(rows);
}

void ms_prepare(g5_ctx* ctx) {
  Graph& g = ctx->graph;
  G5_CHECK(g.built, "g5_batch_prepare: no graph (call g5_construct first)");
  MsState& m = ctx->ms;
  m.release();
  const int64_t rows = g.n_rows;
  m.seen.alloc(rows);
  for (auto& b : m.nz) b.alloc((rows + 63) / 64);
  m.queue.alloc(rows);
  m.prefix.alloc(rows + 1);
  m.chunk_rows.alloc(2 * ((uint64_t)g.nnz / kEpb + 2));
  m.scan_tmp.alloc(scan_tmp_elems(rows + 1));
  m.counters.alloc(kMsCounterWords);
  m.roots.alloc(64);
  m.frp.alloc(G5_MAX_LEVELS);
  if (g.reorder_mode != 0 && g.nnz > 0) {
    // row range of every sweep chunk of the CSR (static for the graph)
    m.sweep_chunks = ((uint64_t)g.nnz + kSweepEpb - 1) / kSweepEpb;
    m.sweep_rows.alloc(2 * m.sweep_chunks);
    hipLaunchKernelGGL(k_chunk_rows<kSweepEpb>, dim3(grid_of((int64_t)(2 * m.sweep_chunks), kBlock, 65536)),
                       dim3(kBlock), 0, ctx->stream, g.offsets.p, rows, m.sweep_chunks, m.sweep_rows.p);
    G5_HIP(hipGetLastError());
  }
  // Every buffer a level may need, sized here so that no batch allocates
  // (the in-loop alloc calls below are then no-ops):
  //   chunk_list / nz_sel  the mixed level's chunk list and selection bitmap
  //   touch                a listed push level has fewer than rows / kTouchBelow frontier edges
  //   miss / ulist         a list-driven tail level follows a level with fewer than
  //                        rows / kListBelow unreached (root, vertex) pairs
  //   fr[0, kMsPreLevels)  the frontier words of the first levels (deeper
  //                        searches add levels as they reach them)
  const int64_t words = (rows + 63) / 64;
  if (m.sweep_chunks) m.chunk_list.alloc(m.sweep_chunks);
  m.nz_sel.alloc(words);
  m.touch.alloc((size_t)((double)rows / kTouchBelow) + 2);
  m.miss.alloc(words);
  m.ulist.alloc((size_t)((double)rows / kListBelow) + 2);
  m.ulist_count.alloc(1);
  for (int l = 0; l < kMsPreLevels; ++l) {
    while ((int)m.fr.size() <= l) m.fr.emplace_back(new DevBuf<uint64_t>());
    m.fr[l]->alloc(rows);
    while ((int)m.fr_dirty.size() <= l) m.fr_dirty.emplace_back(new DevBuf<uint64_t>());
    m.fr_dirty[l]->alloc(words);
  }
  m.fr_exact.assign(m.fr.size(), 0);
  m.fr_count.assign(m.fr.size(), 0);
  if (m.compact_below > 0) ms_alloc_compact(ctx);
  m.h_counters.assign(kMsCounters + T_NUM, 0);
  G5_HIP(hipStreamSynchronize(ctx->stream));  // the published block is reset below
  m.pub.alloc(kMsCounters + T_NUM);
  m.stamps.alloc(T_NUM);
  int khz = 0;
  G5_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device));
  m.clock_khz = khz > 0 ? khz : 100000;
  m.pub_seq = 0;
  m.teps_pub.alloc(65);
  m.teps_seq = 0;
  m.teps_acc.alloc(kTepsStripes * kTepsStride);
  G5_HIP(hipMemsetAsync(m.teps_acc.p, 0, m.teps_acc.bytes(), ctx->stream));
  if (!m.ev0) G5_HIP(hipEventCreate(&m.ev0));
  if (!m.ev1) G5_HIP(hipEventCreate(&m.ev1));
  m.prepared = true;
}

// Level end: the first n_pub counters the host decides the next level with
// are published to coherent host memory, each tagged with the level's
// sequence number, and every counter is cleared for the next level (so no
// fill starts a level).
__global__ void k_ms_publish(unsigned long long* __restrict__ c, int n_pub, Published* __restrict__ p, uint64_t seq,
                             const uint64_t* __restrict__ stamps) {
  if (threadIdx.x < T_NUM) publish(p + kMsCounters + threadIdx.x, wall_clock64() - stamps[threadIdx.x], seq);
  // one thread per counter; counters past the published ones (the per-lane
  // sums of a level that kept none) were not written, but for the list count
  const int n = n_pub > M_NUM ? n_pub : M_NUM + 1;
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    const uint64_t v = ms_stripe_total(c, t);
#pragma unroll 8
    for (int i = 0; i < kMsStripes; ++i) c[i * kMsStride + t] = 0;
    if (t < n_pub) publish(p + t, v, seq);
  }
}

static void ms_wait(MsState& m, int n_pub, hipStream_t s) {
  m.pub.wait(0, n_pub, m.pub_seq, s, "g5_run_bfs_batch: level counters were not published");
  m.pub.wait(kMsCounters, kMsCounters + T_NUM, m.pub_seq, s, "g5_run_bfs_batch: level times were not published");
  for (int i = 0; i < n_pub; ++i) m.h_counters[i] = m.pub.value(i);
  for (int i = kMsCounters; i < kMsCounters + T_NUM; ++i) m.h_counters[i] = m.pub.value(i);
}

static void ms_publish_wait(MsState& m, int n_pub, hipStream_t s) {
  ++m.pub_seq;
  hipLaunchKernelGGL(k_ms_publish, dim3(1), dim3(kBlock), 0, s, (unsigned long long*)m.counters.p, n_pub, m.pub.d,
                     m.pub_seq, m.stamps.p);
  G5_HIP(hipGetLastError());
  ms_wait(m, n_pub, s);
}

// Frontier words of level l, allocated on first use and kept for reuse.
static uint64_t* ms_level(MsState& m, int l, int64_t rows) {
  while ((int)m.fr.size() <= l) m.fr.emplace_back(new DevBuf<uint64_t>());
  const uint64_t* before = m.fr[l]->p;
  m.fr[l]->alloc(rows);
  if ((int)m.fr_exact.size() <= l) {
    m.fr_exact.resize(l + 1, 0);
    m.fr_count.resize(l + 1, 0);
  }
  if (m.fr[l]->p != before) m.fr_exact[l] = 0;  // new memory: contents unknown
  return m.fr[l]->p;
}

// What a level that writes its frontier words sparsely (a push's atomic ORs, a
// listed fold or pull) needs cleared: the words its last run left non-zero
// when those are known and few, else all of them, and where the level only
// sets bits of them the level's own marks.
struct MsClear {
  uint64_t* fr;
  uint64_t* nz;       // the level's marks
  int64_t rows, words;
  int marked;         // fr is non-zero exactly where marked
  int zero_nz;
  uint64_t* stamp;    // of the level, or null
};
// One bitmap word per lane (the marks are read coalesced); a lane zeroes the
// frontier words of its word's set bits.
__device__ __forceinline__ void ms_clear_body(const MsClear& c, int64_t t, int64_t stride) {
  if (c.stamp && t == 0) *c.stamp = wall_clock64();
  if (!c.marked)
    for (int64_t v = t; v < c.rows; v += stride) c.fr[v] = 0;
  for (int64_t wd = t; wd < c.words; wd += stride) {
    if (c.marked)
      for (uint64_t b = c.nz[wd]; b; b &= b - 1) {
        const int64_t v = wd * 64 + __builtin_ctzll(b);
        if (v < c.rows) c.fr[v] = 0;
      }
    if (c.zero_nz) c.nz[wd] = 0;
  }
}

// A level's frontier as a queue: the vertices of `bits` in ascending order,
// and for a push the prefix sums of their degrees and the queue rows of every
// kEpb-edge chunk.  Small ones are made by one workgroup beside the clears of
// the others (k_ms_ready: up to kReadyWords bitmap words and kReadyRows
// vertices); a scan each takes a launch or three, and beyond those sizes one
// workgroup takes longer than they do.
struct MsQueue {
  const uint64_t* bits;
  uint32_t* queue;
  uint64_t* count;     // null: not stored
  uint64_t* prefix;    // null: the queue alone
  int64_t nf;          // vertices, at most (entries past the count add nothing)
  const uint64_t* offsets;
  uint32_t* chunk_rows;
  uint64_t nchunks;    // at most
  uint64_t* bits_out;  // null, or bits again: cleared
};
constexpr int kReadyThreads = 1024;
constexpr int64_t kReadyWords = 16384;
constexpr int kReadyPer = 8;
constexpr int64_t kReadyRows = (int64_t)kReadyThreads * kReadyPer;

__device__ __forceinline__ uint64_t ready_scan(uint64_t v, uint64_t* s_wave, uint64_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t inc = wave_incl_scan(v);
  __syncthreads();
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  uint64_t run = inc - v;
  total = 0;
  for (int w = 0; w < kReadyThreads / 64; ++w) {
    if (w < wave) run += s_wave[w];
    total += s_wave[w];
  }
  return run;
}

__global__ void __launch_bounds__(kReadyThreads) k_ms_ready(MsQueue q, MsClear c) {
  if (blockIdx.x != 0) {
    ms_clear_body(c, (int64_t)(blockIdx.x - 1) * kReadyThreads + threadIdx.x,
                  (int64_t)(gridDim.x - 1) * kReadyThreads);
    return;
  }
  __shared__ uint64_t s_wave[kReadyThreads / 64];
  __shared__ uint64_t s_pre[kReadyRows + 1];
  const int t = threadIdx.x;
  const int64_t per = (c.words + kReadyThreads - 1) / kReadyThreads, w0 = t * per;
  uint64_t n = 0, total, E;
  for (int64_t w = w0; w < w0 + per && w < c.words; ++w) n += (uint64_t)__popcll(q.bits[w]);
  uint64_t at = ready_scan(n, s_wave, total);
  for (int64_t w = w0; w < w0 + per && w < c.words; ++w) {
    for (uint64_t x = q.bits[w]; x; x &= x - 1) q.queue[at++] = (uint32_t)(w * 64 + __builtin_ctzll(x));
    if (q.bits_out) q.bits_out[w] = 0;
  }
  if (t == 0 && q.count) *q.count = total;
  if (!q.prefix) return;
  __syncthreads();  // the queue is read back
  uint64_t d[kReadyPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kReadyPer; ++j) {
    const int64_t i = (int64_t)t * kReadyPer + j;
    d[j] = 0;
    if (i < q.nf && i < (int64_t)total) {
      const uint32_t u = q.queue[i];
      d[j] = q.offsets[u + 1] - q.offsets[u];
    }
    sum += d[j];
  }
  uint64_t run = ready_scan(sum, s_wave, E);
#pragma unroll
  for (int j = 0; j < kReadyPer; ++j) {
    s_pre[t * kReadyPer + j] = run;
    run += d[j];
  }
  if (t == 0) s_pre[kReadyRows] = E;
  __syncthreads();
  for (int64_t i = t; i <= q.nf; i += kReadyThreads) q.prefix[i] = s_pre[i];
  const uint64_t nc = (E + kEpb - 1) / kEpb < q.nchunks ? (E + kEpb - 1) / kEpb : q.nchunks;
  for (uint64_t k = t; k < 2 * nc; k += kReadyThreads) {
    uint64_t key = (k >> 1) * kEpb;
    if (k & 1) key = ((key + kEpb < E) ? key + kEpb : E) - 1;
    int64_t lo = 0, hi = q.nf - 1;  // last row with prefix <= key
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) >> 1;
      if (s_pre[mid] <= key) lo = mid; else hi = mid - 1;
    }
    q.chunk_rows[k] = (uint32_t)lo;
  }
}

__global__ void __launch_bounds__(kBlock) k_ms_clear_level(MsClear c) {
  ms_clear_body(c, (int64_t)blockIdx.x * kBlock + threadIdx.x, (int64_t)gridDim.x * kBlock);
}

// BitsEmitN that clears the bits it has listed (out: the same words, or null).
struct BitsTakeN {
  BitsEmitN emit;
  uint64_t* out;
  __device__ void operator()(size_t w, uint64_t pre) const {
    emit(w, pre);
    if (out && (int64_t)w < emit.words) out[w] = 0;
  }
};

// The level's queue (see MsQueue) and clears.
static void ms_ready(g5_ctx* ctx, const MsQueue& q, const MsClear& c, hipStream_t s) {
  MsState& m = ctx->ms;
  const int64_t items = c.marked ? c.words : c.rows;
  if (c.words <= kReadyWords && q.nf <= kReadyRows) {
    hipLaunchKernelGGL(k_ms_ready, dim3(1 + grid_of(items, kReadyThreads, 255)), dim3(kReadyThreads), 0, s, q, c);
    G5_HIP(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(k_ms_clear_level, dim3(grid_of(items, kBlock, 8192)), dim3(kBlock), 0, s, c);
  device_scan(BitsCountN{q.bits, c.words}, BitsTakeN{{q.bits, c.words, q.queue, m.ulist_count.p}, q.bits_out},
              (size_t)c.words + 1, m.scan_tmp.p, s);
  if (q.prefix) {
    device_scan(FrontierDegreeN{q.queue, q.offsets, m.ulist_count.p}, StoreU64{q.prefix}, (size_t)q.nf + 1,
                m.scan_tmp.p, s);
    if (q.nchunks)
      hipLaunchKernelGGL(k_chunk_rows<kEpb>, dim3(grid_of((int64_t)(2 * q.nchunks), kBlock, 65536)), dim3(kBlock), 0,
                         s, q.prefix, q.nf, q.nchunks, q.chunk_rows);
  }
  G5_HIP(hipGetLastError());
}

// Level l's nonzero bitmap (one bit per vertex whose frontier word is not
// zero), kept per level: it marks the words the level's next run clears.
static uint64_t* ms_marks(MsState& m, int l, int64_t words) {
  while ((int)m.fr_dirty.size() <= l) m.fr_dirty.emplace_back(new DevBuf<uint64_t>());
  m.fr_dirty[l]->alloc(words);
  return m.fr_dirty[l]->p;
}

// Host-driven levels from level l0 on (counters of level l0 - 1 in live /
// nz / fdeg, reached pairs so far in reached): one or more launches per
// level, whose counters the host reads from coherent host memory (the
// counters are clear when it is called).
static void ms_host_levels(g5_ctx* ctx, int l0, uint64_t live, uint64_t nz, uint64_t fdeg, double reached,
                           double roots_live) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  hipStream_t s = ctx->stream;
  const int64_t rows = g.n_rows;
  const int64_t words = (rows + 63) / 64;
  unsigned long long* cnt = (unsigned long long*)m.counters.p;
  g5_batch_stats& st = m.stats;
  const double push_limit = (double)g.nnz / m.alpha;
  const double sweep_limit = m.sweep_below * roots_live * (double)rows;
  const double total_pairs = roots_live * (double)rows;
  const double unseen_frac = m.beta > 0 ? 1.0 / m.beta : 0.0;
  // per-root rule (from the first level, reorder modes 1 and 2): each root's
  // frontier edges and the edges of the vertices it has reached
  const bool lanes_mode = m.lane_rule == 1 && m.sweep_chunks && l0 == 1;
  m.level_masks = lanes_mode;
  double lane_fd[64] = {}, lane_vd[64] = {};
  uint64_t pulled = 0;   // roots that have pulled: they pull from then on
  uint64_t waiting = 0;  // roots over their own threshold that pushed the last level
  const uint64_t* h_lane = m.h_counters.data() + kMsLanes;
  unsigned* d_list_count = (unsigned*)(cnt + M_NUM);
  // turns of a pull that takes 16 rows each up to `limit` words
  m.ulist_count.alloc(1);
  const auto pull_turns = [&](int64_t limit) { return m.pull_unroll == 0 && words <= limit ? words * 4 : words; };
  bool have_miss = false;  // m.miss holds the vertices still missing a live root
  int l = l0 - 1;
  while (live) {
    ++l;
    bool list_level = false;  // this level writes m.miss
    G5_CHECK(l < G5_MAX_LEVELS - 1, "g5_run_bfs_batch: more than 254 levels (uint8 level arrays)");
    uint64_t* next = ms_level(m, l, rows);
    const uint64_t* front = m.fr[l - 1]->p;  // after ms_level: the vector may have grown
    // whether the marks describe this level's frontier words; unset until
    // the level has been enqueued whole (an error midway leaves them unset)
    const bool marked = m.fr_exact[l] != 0;
    m.fr_exact[l] = 0;
    // each level's nonzero bitmap stays with its frontier words (fr_dirty)
    // for the next batch's clear of them
    uint64_t* nz_next = ms_marks(m, l, words);
    const uint64_t* nz_front = m.fr_dirty[l - 1]->p;
    // (a dense mark set is cleared faster by a plain fill)
    uint64_t* const stamp = m.stamps.p + T_LEVEL;
    const auto clear = [&](bool zero_nz, bool first) {
      return MsClear{next, nz_next, rows, words, marked && m.fr_count[l] * 16 < rows ? 1 : 0, zero_nz ? 1 : 0,
                     first ? stamp : nullptr};
    };
    bool push = (double)fdeg < push_limit && total_pairs - reached >= unseen_frac * total_pairs;
    bool sweep = !push && m.sweep_chunks && reached < sweep_limit;
    uint64_t td = 0, bu = 0;
    bool lane_stats = false;  // this level's epilogue gathers per-root statistics
    if (lanes_mode) {
      // pull when the frontier's edges exceed 1/alpha of the edges not yet
      // reached (the roots' own level pushes; all pull in the beta tail); a
      // root that has pulled keeps pulling, so once every live root pulls
      // the level is a plain pull with no per-root statistics
      // A level pulls only when the union of the frontiers has edges enough:
      // a pull reads the rows of everything unreached however few roots it is
      // for, a push the union's rows (S26, 2 of 64 roots over the line at 3 %
      // of the edges: pull 4.7 ms, push of all 1.6; the least a pull pays at
      // is 1/8 of the edges, at larger alpha 16/alpha).  Below kUnionFrom
      // entries a root that has waited a level for that pulls.
      const bool tail = total_pairs - reached < unseen_frac * total_pairs;
      const bool enough = (double)fdeg * std::max(8.0, m.alpha / 16.0) > (double)g.nnz;
      const uint64_t waited = g.nnz < kUnionFrom ? waiting : 0;
      waiting = 0;
      for (int r = 0; r < 64; ++r) {
        const uint64_t bit = UINT64_C(1) << r;
        if (!(live & bit)) continue;
        const double unreached = (double)g.nnz - lane_vd[r];
        const bool over = l > 1 && lane_fd[r] * m.alpha > unreached;
        const bool pull_r = tail || ((pulled | waited) & bit) || (over && enough);
        (pull_r ? bu : td) |= bit;
        if (over && !pull_r) waiting |= bit;
      }
      pulled |= bu;
      push = bu == 0;
      sweep = false;
      lane_stats = td != 0;
    }
    m.level_push[l] = push ? live : td;
    m.level_pull[l] = push ? 0 : (lanes_mode ? bu : live);
    // statistics for the roots still choosing (a root that pulled keeps pulling)
    const LaneEpi lepi{cnt + kMsLanes, g.offsets.p, lanes_mode ? td : live};
    if (lanes_mode && td && bu) {
      // the pushing roots first, then the pull of the others, merging the
      // pushed lanes
      m.nz_sel.alloc(words);
      hipLaunchKernelGGL(k_ms_select, dim3(grid_of(words, kBlock / 64, 8192)), dim3(kBlock), 0, s, front, rows, td,
                         m.nz_sel.p, stamp);
      if (m.mixed_push == 1) {
        // the pushing roots' frontier vertices as a queue (the count stays on
        // the device), their rows as one edge-balanced virtual edge list; the
        // host sizes the scans and grids by the per-root counts of the
        // previous level (the union is at most their sum)
        double nf_ub = 0, fd_ub = 0;
        for (uint64_t x = td; x; x &= x - 1) {
          nf_ub += (double)h_lane[__builtin_ctzll(x)];
          fd_ub += lane_fd[__builtin_ctzll(x)];
        }
        const int64_t nf = (int64_t)std::min<double>(nf_ub, (double)rows);
        const uint64_t E_ub = (uint64_t)std::min<double>(fd_ub, (double)g.nnz);
        const uint64_t nchunks = (E_ub + kEpb - 1) / kEpb;
        G5_CHECK(2 * nchunks <= m.chunk_rows.n, "g5_run_bfs_batch: chunk table too small");
        ms_ready(ctx, MsQueue{m.nz_sel.p, m.queue.p, m.ulist_count.p, m.prefix.p, nf, g.offsets.p, m.chunk_rows.p,
                              nchunks, nullptr}, clear(false, false), s);
        if (nchunks)
          hipLaunchKernelGGL(k_ms_push, dim3(grid_of((int64_t)E_ub, kEpb, 8192)), dim3(kBlock), 0, s, m.queue.p, nf,
                             m.prefix.p, m.chunk_rows.p, g.offsets.p, g.cols.p, front, next, td);
      } else {
        // over the CSR chunks holding one of the pushing roots' frontier vertices
        hipLaunchKernelGGL(k_ms_clear_level, dim3(grid_of(clear(false, false).marked ? words : rows, kBlock, 8192)), dim3(kBlock),
                           0, s, clear(false, false));
        m.chunk_list.alloc(m.sweep_chunks);
        hipLaunchKernelGGL(k_ms_collect, dim3(grid_of((int64_t)m.sweep_chunks, kBlock, 4096)), dim3(kBlock), 0, s,
                           m.sweep_rows.p, m.sweep_chunks, m.nz_sel.p, m.chunk_list.p, d_list_count);
        hipLaunchKernelGGL(k_ms_push_list, dim3(grid_of((int64_t)m.sweep_chunks, 1, 4096)), dim3(kBlock), 0, s,
                           m.chunk_list.p, (const unsigned*)d_list_count, m.sweep_rows.p, (uint64_t)g.nnz,
                           g.offsets.p, g.cols.p, front, m.nz_sel.p, next, td);
      }
      G5_HIP(hipGetLastError());
      // probe unrolling as in the plain pull (pull_unroll)
      decltype(&k_ms_pull_lanes<4, 2>) kpl = k_ms_pull_lanes<4, 2>;
      switch (m.pull_unroll) {
        case 1: kpl = k_ms_pull_lanes<8, 2>; break;
        case 2: kpl = k_ms_pull_lanes<8, 4>; break;
        case 3: kpl = k_ms_pull_lanes<4, 4>; break;
        case 4: kpl = k_ms_pull_lanes<2, 1>; break;
        case 5: kpl = k_ms_pull_lanes<1, 1>; break;
        case 6: kpl = k_ms_pull_lanes<2, 2>; break;
        case 7: kpl = k_ms_pull_lanes<1, 2>; break;
        default: if (words <= kPartWordsFirst) kpl = k_ms_pull_lanes<4, 2, 16>;
      }
      hipLaunchKernelGGL(kpl, dim3(grid_of(pull_turns(kPartWordsFirst), kBlock / 64, m.pull_grid)), dim3(kBlock), 0, s, m.seen.p, front,
                         nz_front, next, nz_next, g.first_nbr.p, g.offsets.p, g.cols.p, rows, bu,
                         m.pull_filter == 1 ? 1 : 0, 1, cnt, lepi);
    } else if (push) {
      const int64_t nf = (int64_t)nz;
      const uint64_t nchunks = (fdeg + kEpb - 1) / kEpb;
      G5_CHECK(2 * nchunks <= m.chunk_rows.n, "g5_run_bfs_batch: chunk table too small");
      // a push whose frontier edges are few next to the rows lists what it
      // touches, and only those vertices are folded
      const uint64_t touch_cap = std::min<uint64_t>(fdeg, (uint64_t)rows);
      const bool touch = (double)fdeg * kTouchBelow < (double)rows;
      ms_ready(ctx, MsQueue{nz_front, m.queue.p, m.ulist_count.p, m.prefix.p, nf, g.offsets.p, m.chunk_rows.p,
                            nchunks, nullptr}, clear(touch, true), s);
      if (touch) {
        m.touch.alloc(std::max<uint64_t>(touch_cap, 1));
        unsigned long long* touch_count = cnt + M_NUM;  // cleared with the counters
        hipLaunchKernelGGL(k_ms_push_touch, dim3(grid_of((int64_t)fdeg, kEpb, 2048)), dim3(kBlock), 0, s,
                           m.queue.p, nf, m.prefix.p, m.chunk_rows.p, g.offsets.p, g.cols.p, front, next, m.touch.p,
                           touch_count);
        hipLaunchKernelGGL(k_ms_finish_list, dim3(grid_of((int64_t)touch_cap, kBlock, 8192)), dim3(kBlock), 0, s,
                           m.seen.p, next, nz_next, g.offsets.p, m.touch.p, (const unsigned long long*)touch_count,
                           cnt, lepi, lane_stats ? 1 : 0);
      } else {
        hipLaunchKernelGGL(k_ms_push, dim3(grid_of((int64_t)fdeg, kEpb, 8192)), dim3(kBlock), 0, s, m.queue.p,
                           nf, m.prefix.p, m.chunk_rows.p, g.offsets.p, g.cols.p, front, next, ~UINT64_C(0));
      }
      G5_HIP(hipGetLastError());
      if (touch) {
        // folded above
      } else if (lane_stats)
        hipLaunchKernelGGL(k_ms_finish_lanes, dim3(grid_of(words, kBlock / 64, 8192)), dim3(kBlock), 0, s, m.seen.p,
                           next, nz_next, g.offsets.p, rows, cnt, lepi);
      else
        hipLaunchKernelGGL(k_ms_finish, dim3(grid_of(words, kBlock / 64, 8192)), dim3(kBlock), 0, s, m.seen.p,
                           next, nz_next, g.offsets.p, rows, cnt);
    } else if (sweep) {
      hipLaunchKernelGGL(k_ms_stamp, dim3(1), dim3(64), 0, s, stamp);
      hipLaunchKernelGGL(k_ms_sweep_clear, dim3(grid_of((int64_t)m.sweep_chunks, kBlock, 4096)), dim3(kBlock), 0,
                         s, m.sweep_rows.p, m.sweep_chunks, g.offsets.p, next);
      hipLaunchKernelGGL(k_ms_sweep, dim3(grid_of((int64_t)m.sweep_chunks, 1, m.sweep_grid)), dim3(kBlock), 0, s,
                         m.sweep_rows.p, (uint64_t)g.nnz, g.offsets.p, g.cols.p, front, nz_front, next);
      G5_HIP(hipGetLastError());
      hipLaunchKernelGGL(k_ms_finish, dim3(grid_of(words, kBlock / 64, 8192)), dim3(kBlock), 0, s, m.seen.p,
                         next, nz_next, g.offsets.p, rows, cnt);
    } else {
      int mode = m.pull_filter == 1 ? kFrontFilter : (m.pull_filter == 2 ? kFrontHybrid : kFrontPlain);
      const uint32_t filter_from = (uint32_t)std::min<double>((double)rows, m.filter_from * (double)rows);
      if (m.compact_below > 0 && (double)nz < m.compact_below * (double)rows) {
        // frontier words of few vertices: pack them densely
        m.pack.alloc(2 * words);
        m.compact.alloc(rows);
        hipLaunchKernelGGL(k_ms_stamp, dim3(1), dim3(64), 0, s, stamp);
        device_scan(CompactCount{nz_front}, CompactEmit{nz_front, front, m.pack.p, m.compact.p}, (size_t)words,
                    m.scan_tmp.p, s);
        mode = kFrontCompact;
      }
      // probe unrolling: (short-row probes per step, long-row probes per lane and step)
      decltype(&k_ms_pull<4, 2>) kp = k_ms_pull<4, 2>;
      switch (m.pull_unroll) {
        case 1: kp = k_ms_pull<8, 2>; break;
        case 2: kp = k_ms_pull<8, 4>; break;
        case 3: kp = k_ms_pull<4, 4>; break;
        case 4: kp = k_ms_pull<2, 1>; break;
        case 5: kp = k_ms_pull<1, 1>; break;
        case 6: kp = k_ms_pull<2, 2>; break;
        case 7: kp = k_ms_pull<1, 2>; break;
        default: if (words <= kPartWords) kp = k_ms_pull<4, 2, 16>;
      }
      // Tail levels: once fewer than rows / kListBelow (root, vertex) pairs
      // are unreached, a pull also marks the vertices still missing a live
      // root (one bit per vertex in m.miss, written 64 at a time), and the
      // next pull takes only those, listed by a scan of the bits (after
      // clearing its frontier array, which must hold zeros elsewhere).
      const double unreached = std::max(0.0, total_pairs - reached);
      if (have_miss && mode == kFrontPlain) {
        const uint64_t ub = (uint64_t)std::min<double>((double)rows, unreached);  // list length bound
        m.ulist.alloc(std::max<uint64_t>(ub, 1));
        ms_ready(ctx, MsQueue{m.miss.p, m.ulist.p, m.ulist_count.p, nullptr, 0, nullptr, nullptr, 0, m.miss.p},
                 clear(true, true), s);
        hipLaunchKernelGGL(k_ms_pull_list, dim3(grid_of((int64_t)ub, kBlock, std::min(m.pull_grid, kListGrid))), dim3(kBlock), 0, s,
                           m.seen.p, front, next, nz_next, g.first_nbr.p, g.offsets.p, g.cols.p, m.ulist.p,
                           m.ulist_count.p, live, m.miss.p, cnt);
        list_level = true;
      } else {
        const bool mark = unreached * kListBelow < (double)rows;
        if (mark) m.miss.alloc(words);
        // the pull writes every word of the level's frontier array (clearing
        // its old words first, one store per marked vertex, so that the pull
        // could skip its zero words, measured no faster)
        hipLaunchKernelGGL(kp, dim3(grid_of(pull_turns(kPartWords), kBlock / 64, m.pull_grid)), dim3(kBlock), 0, s, m.seen.p, front,
                           nz_front, next, nz_next, g.first_nbr.p, g.offsets.p, g.cols.p, rows, live, mode,
                           m.pack.p, m.compact.p, filter_from, cnt, mark ? m.miss.p : nullptr,
                           mode == kFrontCompact ? nullptr : stamp);
        list_level = mark;
      }
    }
    G5_HIP(hipGetLastError());
    m.fr_exact[l] = 1;  // every level form leaves next non-zero exactly at the bits of nz_next
    ms_publish_wait(m, lane_stats ? kMsCounters : M_NUM, s);
    st.direction[l] = (lanes_mode && td && bu) ? 3 : (push ? 1 : (sweep ? 2 : 0));
    if (lane_stats)
      for (int r = 0; r < 64; ++r) {
        lane_fd[r] = (double)h_lane[64 + r];
        lane_vd[r] += (double)h_lane[64 + r];
      }
    have_miss = list_level;  // the next pull level can take the listed vertices only
    st.pairs[l] = (int64_t)m.h_counters[M_PAIRS];
    reached += (double)m.h_counters[M_PAIRS];
    st.num_levels = l + 1;
    st.level_ms[l] = (double)m.h_counters[kMsCounters + T_LEVEL] / (double)m.clock_khz;
    live = m.h_counters[M_LIVE];
    nz = m.h_counters[M_NZ];
    m.fr_count[l] = (int64_t)nz;
    fdeg = m.h_counters[M_FDEG];
  }
}

// Sets up (once per graph and tuning) the persistent path's buffers and the
// hipGraph holding the clears, the root placement and the persistent launch.
static void ms_persistent_setup(g5_ctx* ctx) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  hipStream_t s = ctx->stream;
  const int64_t rows = g.n_rows;
  const int64_t words = (rows + 63) / 64;
  const int K = m.persist_levels;
  if (m.graph_exec && m.graph_levels == K && m.graph_alpha == m.alpha && m.graph_sweep == m.sweep_below &&
      m.graph_grid == m.persist_grid && m.graph_waves == m.persist_waves && m.graph_filter == m.pull_filter &&
      m.graph_beta == m.beta)
    return;
  if (m.graph_exec) {
    (void)hipGraphExecDestroy(m.graph_exec);
    m.graph_exec = nullptr;
  }
  std::vector<uint64_t*> lev(K);
  for (int l = 0; l < K; ++l) lev[l] = ms_level(m, l, rows);
  m.p_fr.alloc(K);
  G5_HIP(hipMemcpyAsync(m.p_fr.p, lev.data(), K * sizeof(uint64_t*), hipMemcpyHostToDevice, s));
  G5_HIP(hipStreamSynchronize(s));  // lev is pageable and local
  m.p_cnt.alloc((size_t)K * M_NUM);
  m.p_ts.alloc(K);
  m.p_dir.alloc(K);
  m.p_misc.alloc(4);  // [0]: done level, [3]: active chunk count
  m.p_bar.alloc(sizeof(GridBarrier) / 8);
  m.chunk_list.alloc(m.sweep_chunks);
  if (!m.h_persist) {
    // counters [levels][M_NUM] | clock [levels] | done level + barrier (4) | roots (64)
    G5_HIP(hipHostMalloc((void**)&m.h_persist, ((size_t)G5_MAX_LEVELS * (M_NUM + 2) + 64) * sizeof(uint64_t),
                         hipHostMallocDefault));
  }
  // co-resident grid: occupancy x compute units, capped by the tuning
  int per_cu = 0, cus = 0;
  const void* kern = nullptr;
  switch (m.persist_waves) {
    case 4: kern = (const void*)k_ms_persistent<4>; break;
    case 6: kern = (const void*)k_ms_persistent<6>; break;
    default: kern = (const void*)k_ms_persistent<8>; break;
  }
  G5_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kBlock, 0));
  G5_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  G5_CHECK(per_cu >= 1, "g5_run_bfs_batch: persistent kernel does not fit a compute unit");
  int64_t grid = (int64_t)per_cu * cus;
  G5_CHECK(grid <= (int64_t)kBarGroup * kBarMaxGroups, "g5_run_bfs_batch: persistent grid beyond the barrier's groups");
  if (m.persist_grid > 0 && m.persist_grid < grid) grid = m.persist_grid;
  m.p_grid = (unsigned)grid;

  MsPersistArgs a{};
  a.offsets = g.offsets.p;
  a.cols = g.cols.p;
  a.first_nbr = g.first_nbr.p;
  a.sweep_rows = m.sweep_rows.p;
  a.rows = rows;
  a.nnz = (uint64_t)g.nnz;
  a.sweep_chunks = m.sweep_chunks;
  a.seen = m.seen.p;
  a.fr = m.p_fr.p;
  a.nz0 = m.nz[0].p;
  a.nz1 = m.nz[1].p;
  a.cnt = (unsigned long long*)m.p_cnt.p;
  a.ts = (long long*)m.p_ts.p;
  a.dir = (int*)m.p_dir.p;
  a.done_levels = (int*)m.p_misc.p;
  a.bar = (GridBarrier*)m.p_bar.p;
  a.chunk_list = m.chunk_list.p;
  a.chunk_count = (unsigned*)(m.p_misc.p + 3);
  a.push_limit = (double)g.nnz / m.alpha;
  a.sweep_below = m.sweep_below;
  a.pull_filter = m.pull_filter;
  a.pull_unseen_frac = m.beta > 0 ? 1.0 / m.beta : 0.0;
  a.max_levels = K;
  a.timeout_ticks = (long long)m.clock_khz * 1000LL * 5;  // 5 s per barrier wait

  // The graph: clears and root placement captured from the stream, then the
  // persistent kernel as a cooperative kernel node (the runtime checks that
  // the whole grid is co-resident, which the grid barrier relies on).
  hipGraph_t graph = nullptr;
  G5_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  hipLaunchKernelGGL(k_ms_fill, dim3(grid_of((int64_t)K * M_NUM, kBlock, 64)), dim3(kBlock), 0, s, m.p_cnt.p,
                     (int64_t)K * M_NUM);
  hipLaunchKernelGGL(k_ms_fill, dim3(1), dim3(kBlock), 0, s, m.p_misc.p, (int64_t)4);
  hipLaunchKernelGGL(k_ms_fill, dim3(grid_of((int64_t)(sizeof(GridBarrier) / 8), kBlock, 64)), dim3(kBlock), 0, s,
                     m.p_bar.p, (int64_t)(sizeof(GridBarrier) / 8));
  hipLaunchKernelGGL(k_ms_clear, dim3(grid_of(rows, kBlock, 4096)), dim3(kBlock), 0, s, m.seen.p, lev[0], rows);
  hipLaunchKernelGGL(k_ms_fill, dim3(grid_of(words, kBlock, 1024)), dim3(kBlock), 0, s, m.nz[0].p, words);
  hipLaunchKernelGGL(k_ms_roots, dim3(1), dim3(64), 0, s, g.old2new.p, m.roots.p, 64, rows, g.offsets.p, m.seen.p,
                     lev[0], (unsigned long long*)m.p_cnt.p);
  hipLaunchKernelGGL(k_ms_roots_nz, dim3(1), dim3(64), 0, s, g.old2new.p, m.roots.p, 64, rows, m.nz[0].p);
  const hipError_t le = hipGetLastError();
  const hipError_t ce = hipStreamEndCapture(s, &graph);
  G5_HIP(le);
  G5_HIP(ce);
  static_assert(sizeof(MsPersistArgs) <= sizeof(m.p_args_storage), "argument block too large");
  std::memcpy(m.p_args_storage, &a, sizeof(a));
  size_t nnodes = 0;
  hipError_t ge = hipGraphGetNodes(graph, nullptr, &nnodes);
  std::vector<hipGraphNode_t> deps(nnodes);
  if (ge == hipSuccess && nnodes) ge = hipGraphGetNodes(graph, deps.data(), &nnodes);
  hipGraphNode_t knode = nullptr;
  if (ge == hipSuccess) {
    hipKernelNodeParams kp{};
    kp.func = (void*)kern;
    kp.gridDim = dim3(m.p_grid);
    kp.blockDim = dim3(kBlock);
    kp.sharedMemBytes = 0;
    void* kargs[] = {(void*)m.p_args_storage};
    kp.kernelParams = kargs;
    kp.extra = nullptr;
    ge = hipGraphAddKernelNode(&knode, graph, deps.data(), nnodes, &kp);
  }
  if (ge == hipSuccess) {
    hipLaunchAttributeValue v{};
    v.cooperative = 1;
    ge = hipGraphKernelNodeSetAttribute(knode, hipLaunchAttributeCooperative, &v);
  }
  if (ge != hipSuccess) {
    (void)hipGraphDestroy(graph);
    G5_HIP(ge);
  }
  const hipError_t ie = hipGraphInstantiate(&m.graph_exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  G5_HIP(ie);
  m.graph_levels = K;
  m.graph_alpha = m.alpha;
  m.graph_sweep = m.sweep_below;
  m.graph_grid = m.persist_grid;
  m.graph_waves = m.persist_waves;
  m.graph_filter = m.pull_filter;
  m.graph_beta = m.beta;
}

// One replay of the batch graph; levels beyond the preallocated arrays go on
// in the host loop.
static void ms_run_persistent(g5_ctx* ctx, const int64_t* roots, int nroots) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  hipStream_t s = ctx->stream;
  ms_persistent_setup(ctx);
  // the persistent kernel clears and writes the frontier words of its levels
  // itself: the per-level marks no longer describe them
  std::fill(m.fr_exact.begin(), m.fr_exact.end(), 0);
  const int K = m.persist_levels;
  int64_t* h_roots = (int64_t*)(m.h_persist + (size_t)G5_MAX_LEVELS * (M_NUM + 2));
  for (int r = 0; r < 64; ++r) h_roots[r] = r < nroots ? roots[r] : -1;
  G5_HIP(hipMemcpyAsync(m.roots.p, h_roots, 64 * sizeof(int64_t), hipMemcpyHostToDevice, s));
  G5_HIP(hipEventRecord(m.ev0, s));
  G5_HIP(hipGraphLaunch(m.graph_exec, s));
  uint64_t* h_cnt = m.h_persist;
  int64_t* h_ts = (int64_t*)(m.h_persist + (size_t)G5_MAX_LEVELS * M_NUM);
  uint64_t* h_misc = m.h_persist + (size_t)G5_MAX_LEVELS * (M_NUM + 1);
  G5_HIP(hipMemcpyAsync(h_cnt, m.p_cnt.p, (size_t)K * M_NUM * 8, hipMemcpyDeviceToHost, s));
  G5_HIP(hipMemcpyAsync(h_ts, m.p_ts.p, (size_t)K * 8, hipMemcpyDeviceToHost, s));
  G5_HIP(hipMemcpyAsync(h_misc, m.p_misc.p, 4 * 8, hipMemcpyDeviceToHost, s));
  GridBarrier* hb = (GridBarrier*)(h_misc + 4);
  G5_HIP(hipMemcpyAsync(hb, m.p_bar.p, 16, hipMemcpyDeviceToHost, s));
  std::vector<int> h_dir(K);
  G5_HIP(hipMemcpyAsync(h_dir.data(), m.p_dir.p, (size_t)K * sizeof(int), hipMemcpyDeviceToHost, s));
  G5_HIP(hipStreamSynchronize(s));

  G5_CHECK_CODE(!hb->abort, G5_ERR_HIP,
                "g5_run_bfs_batch: a grid barrier of the persistent kernel timed out (blocks not co-resident?)");
  const int done = (int)(int32_t)(h_misc[0] & 0xFFFFFFFFu);
  g5_batch_stats& st = m.stats;
  const double tick_ms = 1.0 / (double)m.clock_khz;
  double reached = (double)__builtin_popcountll(h_cnt[M_LIVE]);
  const double roots_live = reached;
  for (int l = 1; l <= done; ++l) {
    st.direction[l] = h_dir[l];
    st.pairs[l] = (int64_t)h_cnt[(size_t)l * M_NUM + M_PAIRS];
    st.level_ms[l] = (double)(h_ts[l] - h_ts[l - 1]) * tick_ms;
    reached += (double)st.pairs[l];
  }
  st.num_levels = done + 1;
  st.persistent_grid = (int32_t)m.p_grid;
  st.persistent_levels = done;
  const uint64_t* last = h_cnt + (size_t)done * M_NUM;
  if (last[M_LIVE]) {
    // out of preallocated levels: continue level by level from the host,
    // which reads the last level's nonzero bitmap from its per-level slot
    const int64_t words = (g.n_rows + 63) / 64;
    G5_HIP(hipMemcpyAsync(ms_marks(m, done, words), m.nz[done & 1].p, words * 8, hipMemcpyDeviceToDevice, s));
    G5_HIP(hipMemsetAsync(m.counters.p, 0, kMsCounterWords * 8, s));  // the host levels expect them clear
    ms_host_levels(ctx, done + 1, last[M_LIVE], last[M_NZ], last[M_FDEG], reached, roots_live);
  }
  (void)g;
}

void ms_run(g5_ctx* ctx, const int64_t* roots, int nroots) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  G5_CHECK(m.prepared, "g5_run_bfs_batch: call g5_batch_prepare first");
  G5_CHECK(nroots >= 1 && nroots <= 64, "g5_run_bfs_batch: 1 to 64 roots per batch");
  for (int r = 0; r < nroots; ++r)
    G5_CHECK(roots[r] >= 0 && roots[r] < g.n, "g5_run_bfs_batch: root out of range");
  hipStream_t s = ctx->stream;
  const int64_t rows = g.n_rows;
  unsigned long long* cnt = (unsigned long long*)m.counters.p;
  m.have_result = false;
  m.level_masks = false;
  m.nroots = nroots;
  m.host_roots.assign(roots, roots + nroots);
  g5_batch_stats& st = m.stats;
  st = g5_batch_stats{};
  st.num_roots = nroots;
  st.num_levels = 1;

  if (m.persistent && m.sweep_chunks) {
    ms_run_persistent(ctx, roots, nroots);
    G5_HIP(hipEventRecord(m.ev1, s));
    G5_HIP(hipEventSynchronize(m.ev1));
    float ms = 0;
    G5_HIP(hipEventElapsedTime(&ms, m.ev0, m.ev1));
    st.device_ms = ms;
  } else {
    uint64_t* fr0 = ms_level(m, 0, rows);
    const int64_t words = (rows + 63) / 64;
    uint64_t* nz0 = ms_marks(m, 0, words);
    MsRoots mr{};
    mr.n = nroots;
    std::copy(roots, roots + nroots, mr.root);
    const bool marked = m.fr_exact[0] != 0;  // by the previous batch's roots
    m.fr_exact[0] = 0;
    hipLaunchKernelGGL(k_ms_begin, dim3(grid_of(rows, kBlock, 4096)), dim3(kBlock), 0, s, m.seen.p, fr0, nz0, rows,
                       words, marked ? 1 : 0, cnt, m.stamps.p);
    ++m.pub_seq;
    hipLaunchKernelGGL(k_ms_place, dim3(1), dim3(64), 0, s, g.old2new.p, mr, rows, g.offsets.p, m.seen.p, fr0, nz0,
                       m.pub.d, m.pub_seq, m.stamps.p);
    G5_HIP(hipGetLastError());
    m.fr_exact[0] = 1;
    m.fr_count[0] = nroots;
    ms_wait(m, M_NUM, s);
    const uint64_t live = m.h_counters[M_LIVE];
    const double roots_live = (double)__builtin_popcountll(live);
    ms_host_levels(ctx, 1, live, m.h_counters[M_NZ], m.h_counters[M_FDEG], roots_live, roots_live);
    st.device_ms = (double)m.h_counters[kMsCounters + T_BATCH] / (double)m.clock_khz;
  }
  m.nlevels = st.num_levels - 1 > 0 ? st.num_levels - 1 : 1;  // levels with frontier words 0..L-1
  m.have_result = true;
}

static void ms_upload_level_ptrs(MsState& m, int nlev, hipStream_t s) {
  std::vector<const uint64_t*> h(nlev);
  for (int i = 0; i < nlev; ++i) h[i] = m.fr[i]->p;
  G5_HIP(hipMemcpyAsync(m.frp.p, h.data(), nlev * sizeof(void*), hipMemcpyHostToDevice, s));
}

// From this many rows on a lane's levels are made by row first: below, the
// levels' frontier words (8 B per row) fit the L2s and one launch is less
// (one lane of S17: 21 us directly, 23 by row; S19, 335k rows: 32 both; S22,
// by row: 112, and 162 with one id per thread and a copy behind it).
constexpr int64_t kRowLevelsFrom = 1 << 19;

void ms_get_levels(g5_ctx* ctx, int lane, uint8_t* host_levels) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  hipStream_t s = ctx->stream;
  G5_CHECK(m.have_result, "g5_batch_get_levels: no batch result");
  G5_CHECK(lane >= 0 && lane < m.nroots, "g5_batch_get_levels: lane out of range");
  LevelWords lw{};
  lw.n = m.stats.num_levels;  // frontier words exist for levels 0..num_levels-1
  for (int i = 0; i < lw.n && i < kMsArgLevels; ++i) {
    lw.fr[i] = m.fr[i]->p;
    lw.nz[i] = m.fr_exact[i] ? m.fr_dirty[i]->p : nullptr;
  }
  if (lw.n > kMsArgLevels) {
    ms_upload_level_ptrs(m, lw.n, s);
    lw.more = (const uint64_t* const*)m.frp.p;
  }
  HostOut out(host_levels, (size_t)g.n, ctx->stage, ctx->bfs.level_out, s);
  if (g.n_rows < kRowLevelsFrom) {
    hipLaunchKernelGGL(k_ms_levels, dim3(grid_of((g.n + 3) / 4, kBlock, 4096)), dim3(kBlock), 0, s, g.old2new.p, g.n,
                       g.n_rows, lw, lane, m.host_roots[lane], (uint8_t*)out.p);
    G5_HIP(hipGetLastError());
  } else {
    m.row_level.alloc(g.n_rows);
    hipLaunchKernelGGL(k_ms_row_levels, dim3(grid_of((g.n_rows + 3) / 4, kBlock, 8192)), dim3(kBlock), 0, s, lw,
                       g.n_rows, lane, m.row_level.p);
    G5_HIP(hipGetLastError());
    launch_make_levels(g.old2new.p, m.row_level.p, g.n, g.n_rows, m.host_roots[lane], (uint8_t*)out.p, s);
  }
  out.finish();
}

void ms_teps_edges(g5_ctx* ctx, int64_t* out) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  G5_CHECK(m.have_result, "g5_batch_teps_edges: no batch result");
  hipStream_t s = ctx->stream;
  const uint64_t all = m.nroots == 64 ? ~UINT64_C(0) : ((UINT64_C(1) << m.nroots) - 1);
  ++m.teps_seq;
  hipLaunchKernelGGL(k_ms_teps, dim3(grid_of((g.n_rows + 63) / 64, kBlock / 64, 2048)), dim3(kBlock), 0, s, m.seen.p,
                     g.weight.p, g.n_rows, all, (unsigned long long*)m.teps_acc.p);
  hipLaunchKernelGGL(k_ms_teps_publish, dim3(1), dim3(128), 0, s, (unsigned long long*)m.teps_acc.p, m.teps_pub.d,
                     m.teps_seq);
  G5_HIP(hipGetLastError());
  m.teps_pub.wait(0, 65, m.teps_seq, s, "g5_batch_teps_edges: the sums were not published");
  for (int r = 0; r < m.nroots; ++r) out[r] = (int64_t)((m.teps_pub.value(r) + m.teps_pub.value(64)) / 2);
}

void ms_model_bytes(g5_ctx* ctx, double* per_level, double* total) {
  Graph& g = ctx->graph;
  MsState& m = ctx->ms;
  G5_CHECK(m.have_result, "g5_batch_model_bytes: no batch result");
  hipStream_t s = ctx->stream;
  const int nlev = m.stats.num_levels;
  ms_upload_level_ptrs(m, nlev, s);
  ctx->acc.alloc(65);
  const uint64_t lanes = m.nroots == 64 ? ~UINT64_C(0) : ((UINT64_C(1) << m.nroots) - 1);
  // The batch's output is fr[l] (written at every level, inside the 24 n
  // term); a root's uint8 levels are unpacked from it on request, outside
  // the batch, so no per-(root, vertex) output byte is counted.
  double tot = 0;
  for (int l = 0; l < G5_MAX_LEVELS; ++l)
    if (per_level) per_level[l] = 0;
  for (int l = 1; l < nlev; ++l) {
    G5_HIP(hipMemsetAsync(ctx->acc.p, 0, 8, s));
    const uint64_t pull = m.level_masks ? m.level_pull[l] & lanes : lanes;
    const uint64_t push = m.level_masks ? m.level_push[l] & lanes : 0;
    hipLaunchKernelGGL(k_ms_model, dim3(grid_of(g.n_rows, kBlock, 8192)), dim3(kBlock), 0, s,
                       (const uint64_t* const*)m.frp.p, l, pull, push, g.offsets.p, g.cols.p, g.n_rows,
                       (unsigned long long*)ctx->acc.p);
    G5_HIP(hipGetLastError());
    uint64_t h = 0;
    G5_HIP(hipMemcpyAsync(&h, ctx->acc.p, 8, hipMemcpyDeviceToHost, s));
    G5_HIP(hipStreamSynchronize(s));
    const double b = 24.0 * (double)g.n + (double)h;
    if (per_level) per_level[l] = b;
    tot += b;
  }
  if (total) *total = tot;
}

}  // namespace g5
