// g5_bfs.hip -- single-root direction-optimizing BFS on gfx950.
//
// Reference behaviour restated: BfsBase::run_bfs (mpi/bfs.hpp:2651-2940):
// level-synchronous search that starts top-down, switches to bottom-up when
// the frontier grows beyond n_active/2000 and back to top-down (for good) when
// fewer than n_active/8 vertices remain unvisited (mpi/bfs.hpp:2799-2829,
// constants mpi/parameters.h:87-89).
//
// Kernels (vertex ids are degree-ordered "new" ids, rows [0, n_rows)):
//   top-down   k_td_expand: the frontier's rows are concatenated into one
//              virtual edge list (exclusive scan of frontier degrees); each
//              workgroup takes kEpb-edge chunks, stages the prefix/row-base/
//              source of the frontier vertices overlapping its chunk in LDS and
//              binary-searches there once per lane, so hub rows are split
//              across the whole grid.  Small levels test-and-set the visited
//              bitmap and append winners through LDS (one global atomic per
//              chunk); hub levels use no atomics: the visited bitmap is a
//              read-only snapshot, new targets get level/parent with benign
//              races, and one pass over the level array gives the frontier.
//              While the search grows, a hub level first settles its
//              highest-degree targets bottom-up (k_td_head) and expands only
//              the row suffixes beyond them (k_td_expand_segs).
//              After the bottom-up phase, a top-down level whose frontier is
//              large against the unvisited vertices is found by the bottom-up
//              kernel (same vertices, far fewer probes).
//   steps      k_bfs_step: one launch per level, whose workgroups all apply
//              the switch rule to the last level's counts, so that no level
//              waits for the host; it runs small and mid top-down levels and,
//              on graphs up to kStepMaxWords bitmap words, bottom-up levels.
//   host loop  the other levels: a one-wave kernel publishes the level's
//              counters to coherent host memory, each value tagged with the
//              level's sequence number, where the host reads them for the
//              alpha/beta rule.
//   queues     a top-down frontier that comes from a bitmap is rebuilt by an
//              exclusive scan of per-word popcounts (ascending vertex order).
//   bottom-up  step_bottom_up (in steps and in k_bu): a wave takes up to 16
//              64-vertex bitmap words a turn.  Unvisited vertices first probe
//              their first (highest-degree) neighbour from the coalesced
//              first_nbr array, four words in flight; the rows of those who
//              missed are searched with every lane busy.  The visited snapshot
//              of the previous level is read-only; the next bitmap's words are
//              written once per turn.
#include "g5_answers.hpp"
#include "g5_ctx.hpp"
#include "g5_frontier.hpp"
#include "g5_prims.hpp"

#include <algorithm>

namespace g5 {

constexpr uint64_t kTdSmall = 1 << 20;  // top-down levels up to this many edges use the atomic path
constexpr int kBinShift = 19;           // binned top-down: at least 2^19 targets per bucket
constexpr int kShortRow = 32;    // bottom-up: lane-sequential scan up to this length
// Searches of many rows at a time (kR = 1: k_bu, k_td_head): rows over
// kShortRow1 entries go to groups of 16 lanes, and what kGroupTurns turns
// leave of a very long one to the whole wave.  A wave per row read 64 entries
// where a few decide, one row after another (S26 700 us a search, S28 2,396;
// so 646 and 2,224; with the limit 8 and 32: 644 and 662, 2,244 and 2,190).
constexpr int kShortRow1 = 16;
constexpr int kGroupTurns = 8;
constexpr uint32_t kNoNbr = 0xFFFFFFFFu;

// counters: vertices found; the root (new id); head words (k_td_head_size);
// frontier edges of the next level, summed by a small top-down level.  The
// found and next-edge sums of whole grids go to the stripes behind them
// (words S_FOUND and S_NEXT_E of each); k_publish adds the stripes up.
// C_FOUND itself only hands out queue positions in a small top-down level.
enum { C_FOUND = 0, C_AUX = 1, C_HEAD = 2, C_NEXT_E = 3, C_NUM = 4 };
enum { S_FOUND = 0, S_NEXT_E = 1 };
constexpr int kStripeBase = 8;  // words: the stripes start on a 64-byte line of their own
constexpr int kBfsCounters = kStripeBase + kStripes * kStripeWords;

// Top-down expansion of one level.  The frontier's rows form one virtual edge
// list (prefix = exclusive scan of frontier degrees, E = prefix[nf]); every
// workgroup takes kEpb-edge chunks and each lane walks kEpt consecutive edges.
//   kBulk = false (small levels): test-and-set on the visited bitmap itself
//           (atomicOr after a plain-load filter); winners are staged in LDS
//           and appended to 'next' with one global atomic per chunk, which
//           also counts them in counters[C_FOUND]; their degree sum (the
//           next level's frontier edges) goes to counters[C_NEXT_E].
//   kBulk = true  (hub levels): no atomics: a target gets level and parent
//           unless its level is already set (racing writers store the same
//           level and a valid parent); k_td_finish then takes the exact new
//           set from the level array.  The visited-bitmap snapshot is probed
//           first only when probe_vis is set (levels after the bottom-up
//           phase, where it drops most targets); while the search grows it
//           holds few vertices and the level test alone decides.
// Rows below the returned id were settled by k_td_head (none without a head).
__device__ __forceinline__ uint32_t head_bound(const unsigned long long* head_words) {
  if (!head_words) return 0;
  const unsigned long long v = *head_words * 64;
  return v < UINT32_MAX ? (uint32_t)v : UINT32_MAX;
}

__device__ __forceinline__ void bulk_claims(uint64_t e0, uint64_t e1, int cnt, const ChunkRows& cr,
                                            const uint32_t* __restrict__ cols, const uint64_t* vis,
                                            uint8_t* level, uint32_t* __restrict__ parent, uint32_t lvl,
                                            int probe_vis, uint32_t head) {
  // every probe of the lane's edges in flight before any claim
  uint32_t w[kEpt], u[kEpt];
  bool ok[kEpt];
  gather_strided(e0, e1, cnt, cr, cols, w, u, ok);
  if (probe_vis) {
    // most targets are visited already: the bitmap (1/8 of the level
    // array's footprint) drops them before any level probe
    uint64_t vw[kEpt];
#pragma unroll
    for (int j = 0; j < kEpt; ++j) vw[j] = ok[j] ? vis[w[j] >> 6] : 0;
#pragma unroll
    for (int j = 0; j < kEpt; ++j) ok[j] = ok[j] && !((vw[j] >> (w[j] & 63)) & 1);
  }
  // targets below 'head' were settled by k_td_head
#pragma unroll
  for (int j = 0; j < kEpt; ++j) ok[j] = ok[j] && w[j] >= head;
  uint8_t lv[kEpt];
#pragma unroll
  for (int j = 0; j < kEpt; ++j) lv[j] = ok[j] ? level[w[j]] : 0;
#pragma unroll
  for (int j = 0; j < kEpt; ++j)
    if (ok[j] && lv[j] == 0xFF) {
      level[w[j]] = (uint8_t)lvl;
      parent[w[j]] = u[j];
    }
}

template <bool kBulk>
__global__ void __launch_bounds__(kBlock) k_td_expand(
    const uint32_t* __restrict__ queue, int64_t nf, const uint64_t* __restrict__ prefix,
    const uint32_t* __restrict__ chunk_rows, const uint64_t* __restrict__ offsets,
    const uint32_t* __restrict__ cols, uint64_t* vis, uint8_t* level, uint32_t* __restrict__ parent,
    uint32_t* __restrict__ next, unsigned long long* __restrict__ counters, uint32_t lvl, int probe_vis,
    const unsigned long long* __restrict__ head_words) {
  __shared__ ChunkRows cr;
  __shared__ uint32_t s_q[kBulk ? 1 : kEpb];
  __shared__ uint32_t s_qn;
  __shared__ uint64_t s_qbase;
  const uint64_t E = prefix[nf];
  // both forms are launched before the host knows E; the other one exits
  if (kBulk ? E <= kTdSmall : E > kTdSmall) return;
  const uint32_t head = head_bound(head_words);
  uint64_t next_e = 0;  // degree sum of this lane's winners (small levels)
  for (uint64_t chunk = blockIdx.x; chunk * kEpb < E; chunk += gridDim.x) {
    const uint64_t e0 = chunk * kEpb;
    const uint64_t e1 = (e0 + kEpb < E) ? e0 + kEpb : E;
    if (!kBulk && threadIdx.x == 0) s_qn = 0;
    const int cnt = stage_chunk(chunk, chunk_rows, queue, prefix, offsets, cr);
    const auto visit = [&](uint32_t w, uint32_t u) {
      const uint64_t bit = UINT64_C(1) << (w & 63);
      if (vis[w >> 6] & bit) return;
      const uint64_t old = atomicOr((unsigned long long*)(vis + (w >> 6)), (unsigned long long)bit);
      if (old & bit) return;
      level[w] = (uint8_t)lvl;
      parent[w] = u;
      s_q[atomicAdd(&s_qn, 1u)] = w;
      next_e += offsets[w + 1] - offsets[w];
    };
    if (kBulk) {
      bulk_claims(e0, e1, cnt, cr, cols, vis, level, parent, lvl, probe_vis, head);
    } else {
      walk_strided(e0, e1, cnt, cr, cols, visit);
    }
    if (!kBulk) {
      __syncthreads();
      if (threadIdx.x == 0) s_qbase = s_qn ? atomicAdd(counters + C_FOUND, (unsigned long long)s_qn) : 0;
      __syncthreads();
      for (uint32_t j = threadIdx.x; j < s_qn; j += kBlock) next[s_qbase + j] = s_q[j];
    }
    __syncthreads();
  }
  // the next level's frontier edges, so that the host can skip the launches
  // of the other form there
  if (!kBulk) block_add(next_e, stripe_of(counters + kStripeBase, S_NEXT_E));
}

// --- piece-ordered hub levels ---------------------------------------------
// A hub level's frontier rows hold up to billions of edges whose targets,
// sorted within each row, spread over the whole level array, so taking the
// rows one after another keeps the grid's probes scattered over all of it.
// Instead every row is cut into P pieces by position (piece k of a row of
// degree d holds its positions [k*d/P, (k+1)*d/P)) and pieces are taken piece
// index first.  The rows of a Kronecker graph share nearly one neighbour
// distribution (a target bit is 0 with probability A/(A+B) = 0.75 or
// C/(C+D) = 0.79 for the two values of the row bit under the 0.57/0.19/0.19
// initiator), so the k-th pieces of all rows cover about the same target
// range and the level and parent bytes the grid touches at a time stay
// cache-sized.  One scan compacts the non-empty pieces into a segment list
// (the scanned value carries the piece count above bit 40 and its edges
// below) that the chunked bulk expansion walks like frontier rows.
constexpr int kSegCountShift = 40;
constexpr uint64_t kSegEdgeMask = (UINT64_C(1) << kSegCountShift) - 1;
constexpr int64_t kSegMax = (INT64_C(1) << 24) - 1;  // segments of one level (count field width)

struct PieceLen {
  const uint32_t* queue;
  const uint64_t* offsets;
  const uint64_t* prefix;
  int64_t nf;
  int64_t pieces;
  // piece s = k * nf + i: frontier row i's piece k -> source, first cols index, length
  __device__ void piece(size_t s, uint32_t& u, uint64_t& a, uint64_t& len) const {
    const int64_t k = (int64_t)s / nf, i = (int64_t)s - k * nf;
    u = queue[i];
    const uint64_t o = offsets[u], d = offsets[u + 1] - o;
    a = o + (uint64_t)k * d / (uint64_t)pieces;
    len = o + (uint64_t)(k + 1) * d / (uint64_t)pieces - a;
  }
  __device__ uint64_t operator()(size_t s) const {
    // a small level (E <= kTdSmall) makes no segments
    if ((int64_t)s >= nf * pieces || prefix[nf] <= kTdSmall) return 0;
    uint32_t u;
    uint64_t a, len;
    piece(s, u, a, len);
    return len ? (UINT64_C(1) << kSegCountShift) | len : 0;
  }
};
// Exact target blocks (block = 2^shift consecutive target ids): the first
// hub_rows rows (the highest-degree ones in degree order) carry the cols
// index of their first entry in every block, relative to the row start,
// bnd[v * (nb + 1) + b] for b in [0, nb] (bnd[.. + nb] = degree).  Piece
// s = k * nf + i is row i's block k for a hub row and, for k = nb, the whole
// row of any other frontier vertex (whose edges are few at a hub level).
struct BlockLen {
  const uint32_t* queue;
  const uint64_t* offsets;
  const uint64_t* prefix;
  int64_t nf;
  int64_t pieces;  // nb + 1
  const uint32_t* bnd;
  int64_t hub_rows;
  __device__ void piece(size_t s, uint32_t& u, uint64_t& a, uint64_t& len) const {
    const int64_t k = (int64_t)s / nf, i = (int64_t)s - k * nf;
    u = queue[i];
    const uint64_t o = offsets[u];
    a = o;
    len = 0;
    if ((int64_t)u < hub_rows) {
      if (k + 1 < pieces) {
        const uint32_t* r = bnd + (int64_t)u * pieces + k;
        a = o + r[0];
        len = r[1] - r[0];
      }
    } else if (k + 1 == pieces) {
      len = offsets[u + 1] - o;
    }
  }
  __device__ uint64_t operator()(size_t s) const {
    if ((int64_t)s >= nf * pieces || prefix[nf] <= kTdSmall) return 0;
    uint32_t u;
    uint64_t a, len;
    piece(s, u, a, len);
    return len ? (UINT64_C(1) << kSegCountShift) | len : 0;
  }
};

// bnd of the block index (one lane per row and block; the lanes of a wave
// share a row, so the first steps of their binary searches coincide)
__global__ void __launch_bounds__(kBlock) k_hub_bounds(const uint64_t* __restrict__ offsets,
                                                       const uint32_t* __restrict__ cols, int64_t hub_rows,
                                                       int64_t pieces, int shift, uint32_t* __restrict__ bnd) {
  const int64_t total = hub_rows * pieces;
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < total; t += (int64_t)gridDim.x * kBlock) {
    const int64_t v = t / pieces, b = t - v * pieces;
    const uint64_t key = (uint64_t)b << shift;
    uint64_t lo = offsets[v], hi = offsets[v + 1];
    const uint64_t o = lo;
    while (lo < hi) {  // first entry >= key
      const uint64_t mid = (lo + hi) >> 1;
      if (cols[mid] < key) lo = mid + 1; else hi = mid;
    }
    bnd[t] = (uint32_t)(lo - o);
  }
}

// With a head (k_td_head), the edges a frontier row still has to expand are
// its suffix of targets >= the head bound (rows are sorted): one segment per
// row, whose start k_suffix_start finds by binary search (one lane per row),
// so the expansion no longer reads the columns of edges into the head.
__global__ void __launch_bounds__(kBlock) k_suffix_start(const uint32_t* __restrict__ queue, int64_t nf,
                                                         const uint64_t* __restrict__ prefix,
                                                         const uint64_t* __restrict__ offsets,
                                                         const uint32_t* __restrict__ cols,
                                                         const unsigned long long* __restrict__ head_words,
                                                         uint64_t* __restrict__ start) {
  if (prefix[nf] <= kTdSmall) return;
  const uint32_t h = head_bound(head_words);
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nf; i += (int64_t)gridDim.x * kBlock) {
    const uint32_t u = queue[i];
    uint64_t lo = offsets[u], hi = offsets[u + 1];
    while (lo < hi) {  // first entry >= h
      const uint64_t mid = (lo + hi) >> 1;
      if (cols[mid] < h) lo = mid + 1; else hi = mid;
    }
    start[i] = lo;
  }
}

struct SuffixLen {
  const uint32_t* queue;
  const uint64_t* offsets;
  const uint64_t* prefix;
  int64_t nf;
  int64_t pieces;         // 1
  const uint64_t* start;  // k_suffix_start
  __device__ void piece(size_t s, uint32_t& u, uint64_t& a, uint64_t& len) const {
    u = queue[s];
    a = start[s];
    len = offsets[u + 1] - a;
  }
  __device__ uint64_t operator()(size_t s) const {
    if ((int64_t)s >= nf || prefix[nf] <= kTdSmall) return 0;
    uint32_t u;
    uint64_t a, len;
    piece(s, u, a, len);
    return len ? (UINT64_C(1) << kSegCountShift) | len : 0;
  }
};

template <class Len>
struct PieceEmit {
  Len in;
  uint64_t* seg_pre;   // first virtual edge of each segment; seg_pre[count] = E
  uint64_t* seg_base;  // cols index - seg_pre
  uint32_t* seg_src;
  uint64_t* seg_count;
  __device__ void operator()(size_t s, uint64_t pre) const {
    const uint64_t pos = pre >> kSegCountShift, ep = pre & kSegEdgeMask;
    if ((int64_t)s == in.nf * in.pieces) {  // the extra last element carries the totals
      seg_count[0] = pos;
      seg_pre[pos] = ep;
      return;
    }
    if (in.prefix[in.nf] <= kTdSmall) return;
    uint32_t u;
    uint64_t a, len;
    in.piece(s, u, a, len);
    if (!len) return;
    seg_pre[pos] = ep;
    seg_base[pos] = a - ep;
    seg_src[pos] = u;
  }
};

// k_chunk_rows over the segment list, whose length is known on the device only.
__global__ void __launch_bounds__(kBlock) k_chunk_segs(const uint64_t* __restrict__ seg_pre,
                                                       const uint64_t* __restrict__ seg_count, uint64_t nchunks,
                                                       uint32_t* __restrict__ rows_out) {
  const int64_t ns = (int64_t)seg_count[0];
  if (ns == 0) return;
  const uint64_t E = seg_pre[ns];
  const uint64_t nc = (E + kEpb - 1) / kEpb < nchunks ? (E + kEpb - 1) / kEpb : nchunks;
  for (uint64_t t = (uint64_t)blockIdx.x * kBlock + threadIdx.x; t < 2 * nc; t += (uint64_t)gridDim.x * kBlock) {
    const uint64_t c = t >> 1;
    uint64_t key = c * kEpb;
    if (t & 1) key = ((key + kEpb < E) ? key + kEpb : E) - 1;
    int64_t lo = 0, hi = ns - 1;  // last segment with seg_pre <= key
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) >> 1;
      if (seg_pre[mid] <= key) lo = mid; else hi = mid - 1;
    }
    rows_out[t] = (uint32_t)lo;
  }
}

// The bulk expansion over the segment list: a bulk level (E = prefix[nf] >
// kTdSmall) walks the seg_pre[count] edges of its segments.
__global__ void __launch_bounds__(kBlock) k_td_expand_segs(
    const uint64_t* __restrict__ prefix, int64_t nf, const uint64_t* __restrict__ seg_pre,
    const uint64_t* __restrict__ seg_base, const uint32_t* __restrict__ seg_src,
    const uint64_t* __restrict__ seg_count, const uint32_t* __restrict__ chunk_rows,
    const uint32_t* __restrict__ cols, const uint64_t* vis, uint8_t* level, uint32_t* __restrict__ parent,
    uint32_t lvl, const unsigned long long* __restrict__ head_words) {
  __shared__ ChunkRows cr;
  if (prefix[nf] <= kTdSmall) return;
  const uint64_t E = seg_pre[*seg_count];
  const uint32_t head = head_bound(head_words);
  for (uint64_t chunk = blockIdx.x; chunk * kEpb < E; chunk += gridDim.x) {
    const uint64_t e0 = chunk * kEpb;
    const uint64_t e1 = (e0 + kEpb < E) ? e0 + kEpb : E;
    // every segment is non-empty, so at most kEpb + 1 of them overlap a chunk
    const int64_t i0 = chunk_rows[2 * chunk];
    int cnt = (int)((int64_t)chunk_rows[2 * chunk + 1] - i0 + 1);
    cnt = cnt > kEpb + 1 ? kEpb + 1 : cnt;
    for (int j = threadIdx.x; j < cnt; j += kBlock) {
      cr.pre[j] = seg_pre[i0 + j];
      cr.base[j] = seg_base[i0 + j];
      cr.src[j] = seg_src[i0 + j];
    }
    __syncthreads();
    bulk_claims(e0, e1, cnt, cr, cols, vis, level, parent, lvl, 0, head);
    __syncthreads();
  }
}

// Row part of the bottom-up probe: an entry of [offsets[v] + 1, offsets[v + 1])
// (the first neighbour is probed apart, from the coalesced first_nbr array)
// whose bit is set in bm.  Every lane of the wave calls it; lanes with
// active=false only help.  Rows up to kShortRow are scanned by their lane, kU
// entries a turn; longer rows by the whole wave, kR rows a turn, 64 entries of
// each (the last one left takes all kR x 64), a ballot giving a row's first
// hit; with kR = 1 by groups of 16 lanes first (see kShortRow1).  A turn is a chain of two dependent loads, so on small graphs, whose
// bottom-up levels are a few such chains, the turns are what counts (kU 8, kR
// 4); on large ones the probes past a hit are (kU 4, kR 1 with two per lane).
template <int kU, int kR>
__device__ __forceinline__ bool row_marked_nbr(bool active, uint32_t v, const uint64_t* __restrict__ bm,
                                               const uint64_t* __restrict__ offsets,
                                               const uint32_t* __restrict__ cols, uint32_t& p) {
  const int lane = threadIdx.x & 63;
  bool found = false, need = false;
  uint64_t rb = 0, re = 0;
  if (active) {
    rb = offsets[v] + 1;
    re = offsets[v + 1];
    need = rb < re;
  }
  if (need && re - rb <= (uint64_t)(kR == 1 ? kShortRow1 : kShortRow)) {
    // independent probes (entries past the row repeat the first); any marked
    // neighbour is a valid parent, the first is taken
    for (uint64_t k = rb; k < re && !found; k += kU) {
      uint32_t c[kU];
      c[0] = cols[k];
#pragma unroll
      for (int j = 1; j < kU; ++j) c[j] = k + j < re ? cols[k + j] : c[0];
      bool h[kU];
#pragma unroll
      for (int j = 0; j < kU; ++j) h[j] = bit_set(bm, c[j]);
#pragma unroll
      for (int j = kU - 1; j >= 0; --j)
        if (h[j]) {
          found = true;
          p = c[j];
        }
    }
    need = false;
  }
  uint64_t lm = __ballot(need);
  if (kR == 1) {
    // by groups of 16 lanes, four rows at a time, a group taking the next row
    // as soon as its own is done
    const int gid = lane / 16, gl = lane % 16;
    uint64_t rest = 0;
    int src = -1, turn = 0;
    uint64_t b = 0, e = 0;
    for (;;) {
      const uint64_t idle = __ballot(src < 0);
      if (idle) {
        if (!lm && idle == ~UINT64_C(0)) break;
        const int rank = __popcll(idle & ((UINT64_C(1) << (gid * 16)) - 1)) / 16;
        int take = -1;
        for (int i = 0; i < __popcll(idle) / 16 && lm; ++i) {
          if (i == rank) take = __builtin_ctzll(lm);
          lm &= lm - 1;
        }
        const int from = take < 0 ? lane : take;
        const uint64_t b1 = __shfl(rb, from, 64), e1 = __shfl(re, from, 64);
        if (src < 0 && take >= 0) {
          src = take;
          b = b1;
          e = e1;
          turn = 0;
        }
      }
      const bool in = src >= 0 && b + gl < e;
      const uint32_t c = in ? cols[b + gl] : 0;
      const uint64_t m = __ballot(in && bit_set(bm, c));
      b += 16;
      ++turn;
      const bool done = src >= 0 && (((m >> (gid * 16)) & 0xFFFF) || b >= e);
      const bool pass = src >= 0 && !done && turn >= kGroupTurns && e - b > 128;  // left to the whole wave
      const uint64_t out = __ballot(done || pass);
      if (out) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (!((out >> (g * 16)) & 1)) continue;
          const int s = __builtin_amdgcn_readlane(src, g * 16);
          const uint32_t gm = (uint32_t)(m >> (g * 16)) & 0xFFFF;
          const uint32_t hp = __shfl(c, g * 16 + (gm ? __builtin_ctz(gm) : 0), 64);
          const uint64_t gb = __shfl(b, g * 16, 64);
          if (lane == s) {
            if (gm) {
              found = true;
              p = hp;
            }
            rb = gb;
          }
          rest |= (uint64_t)(__builtin_amdgcn_readlane((int)pass, g * 16) & 1) << s;
        }
        if (done || pass) src = -1;
      }
    }
    lm = rest;
  }
  while (lm) {
    constexpr int kSlots = kR > 1 ? kR : 2;
    int src[kSlots];
    uint64_t b[kSlots], e[kSlots];
    int n = 0;  // rows of this turn
#pragma unroll
    for (int j = 0; j < kR; ++j) {
      src[j] = -1;
      b[j] = e[j] = 0;
      if (lm) {
        src[j] = __builtin_ctzll(lm);
        lm &= lm - 1;
        b[j] = __shfl(rb, src[j], 64);
        e[j] = __shfl(re, src[j], 64);
        ++n;
      }
    }
    while (n > 1) {  // 64 entries of every row
      uint32_t c[kR];
      bool h[kR];
#pragma unroll
      for (int j = 0; j < kR; ++j) c[j] = b[j] + lane < e[j] ? cols[b[j] + lane] : 0;
#pragma unroll
      for (int j = 0; j < kR; ++j) h[j] = b[j] + lane < e[j] && bit_set(bm, c[j]);
#pragma unroll
      for (int j = 0; j < kR; ++j) {
        if (b[j] >= e[j]) continue;
        const uint64_t m = __ballot(h[j]);
        if (m) {
          const uint32_t hp = __shfl(c[j], __builtin_ctzll(m), 64);
          if (lane == src[j]) {
            found = true;
            p = hp;
          }
        }
        b[j] = m ? e[j] : b[j] + 64;
        if (b[j] >= e[j]) --n;
      }
    }
    if (n == 1) {  // one row: all slots
      int s1 = -1;
      uint64_t b1 = 0, e1 = 0;
#pragma unroll
      for (int j = 0; j < kR; ++j)
        if (b[j] < e[j]) {
          s1 = src[j];
          b1 = b[j];
          e1 = e[j];
        }
      for (; b1 < e1; b1 += 64 * kSlots) {
        uint32_t c[kSlots];
        bool h[kSlots];
#pragma unroll
        for (int j = 0; j < kSlots; ++j) c[j] = b1 + 64 * j + lane < e1 ? cols[b1 + 64 * j + lane] : 0;
#pragma unroll
        for (int j = 0; j < kSlots; ++j) h[j] = b1 + 64 * j + lane < e1 && bit_set(bm, c[j]);
        uint32_t hp = 0;
        bool any = false;
#pragma unroll
        for (int j = kSlots - 1; j >= 0; --j) {
          const uint64_t m = __ballot(h[j]);
          if (m) {
            any = true;
            hp = __shfl(c[j], __builtin_ctzll(m), 64);
          }
        }
        if (any) {
          if (lane == s1) {
            found = true;
            p = hp;
          }
          break;
        }
      }
    }
  }
  return found;
}

// First neighbour of v, in ascending (highest degree first) order, whose bit
// is set in bm: the bottom-up probe (first_nbr, then the row).  Every lane of
// the wave calls it; lanes with active=false only help.
__device__ __forceinline__ bool first_marked_nbr(bool active, uint32_t v, const uint64_t* __restrict__ bm,
                                                 const uint32_t* __restrict__ first_nbr,
                                                 const uint64_t* __restrict__ offsets,
                                                 const uint32_t* __restrict__ cols, uint32_t& p) {
  const uint32_t f = active ? first_nbr[v] : kNoNbr;
  const bool hit = f != kNoNbr && bit_set(bm, f);
  if (hit) p = f;
  const bool more = row_marked_nbr<4, 1>(f != kNoNbr && !hit, v, bm, offsets, cols, p);
  return hit || more;
}

// Head of a growing bulk top-down level: the rows [0, 64 * head_words) (the
// highest-degree vertices in degree order) are settled bottom-up before the
// expansion, which then skips every edge into them.  An unvisited vertex
// whose neighbour is visited is reached at this level, because a neighbour
// from an older level would have reached it earlier, so the visited bitmap
// stands for the frontier and the vertex gets the same level it would get
// top-down, with a valid parent.  The hubs' rows are long, but most of them
// meet a visited neighbour within their first (highest-degree) entries,
// whereas top-down every frontier row probes them again and again.
__global__ void __launch_bounds__(kBlock) k_td_head(const uint64_t* __restrict__ vis,
                                                    const uint32_t* __restrict__ first_nbr,
                                                    const uint64_t* __restrict__ offsets,
                                                    const uint32_t* __restrict__ cols, uint8_t* __restrict__ level,
                                                    uint32_t* __restrict__ parent,
                                                    const unsigned long long* __restrict__ head_words_p, uint32_t lvl) {
  const int64_t head_words = (int64_t)*head_words_p;  // 0 at a small level
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (kBlock / 64);
  for (int64_t w = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); w < head_words; w += nwaves) {
    const uint64_t cur = vis[w];
    if (cur == ~UINT64_C(0)) continue;
    const uint32_t v = (uint32_t)(w * 64 + lane);
    uint32_t p = 0;
    if (first_marked_nbr(!((cur >> lane) & 1), v, vis, first_nbr, offsets, cols, p)) {
      level[v] = (uint8_t)lvl;
      parent[v] = p;
    }
  }
}

// How far the head reaches, from the level's frontier edge count E: a row
// of degree d belongs to it when d >= factor * (nnz / E)^2.  Settling such a
// vertex bottom-up takes about nnz / E probes (a random neighbour is a
// frontier vertex with probability about E / nnz), while top-down its
// level byte is probed about d * E / nnz times; the two balance at
// d = (nnz / E)^2.  Rows are in descending degree order, so the head is the
// prefix of rows above the threshold (found by binary search), in bitmap
// words.  A small level (E <= kTdSmall) gets none.
__global__ void k_td_head_size(const uint64_t* __restrict__ prefix, int64_t nf,
                               const uint64_t* __restrict__ offsets, int64_t rows, int64_t words, double nnz,
                               double factor, unsigned long long* __restrict__ head_words) {
  const uint64_t E = prefix[nf];
  int64_t h = 0;
  if (E > kTdSmall) {
    const double r = nnz / (double)E;
    const double thr = factor * r * r;
    int64_t lo = 0, hi = rows;  // first row with degree < thr
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if ((double)(offsets[mid + 1] - offsets[mid]) >= thr) lo = mid + 1; else hi = mid;
    }
    h = (lo + 63) / 64;
    if (h > words) h = words;
  }
  *head_words = (unsigned long long)h;
}

// Binned top-down for hub levels (hundreds of millions of frontier edges):
// the edges' (target, source) pairs are first written out grouped by
// target range (bucket = target >> shift, 2^shift targets, whose level and
// parent bytes fit in L2), then applied bucket after bucket, so the
// random level probes of the plain bulk path become L2-local.  Two passes
// over the frontier's rows (count, then scatter with per-block ranges
// reserved by one atomic per bucket) and one over the pairs.
constexpr int kBinMaxBuckets = 2048;

__global__ void __launch_bounds__(kBlock) k_td_bin_count(const uint32_t* __restrict__ queue, int64_t nf,
                                                         const uint64_t* __restrict__ prefix,
                                                         const uint32_t* __restrict__ chunk_rows,
                                                         const uint64_t* __restrict__ offsets,
                                                         const uint32_t* __restrict__ cols, int shift, int nb,
                                                         unsigned long long* __restrict__ bucket_cnt) {
  __shared__ ChunkRows cr;
  __shared__ unsigned s_hist[kBinMaxBuckets];
  for (int i = threadIdx.x; i < nb; i += kBlock) s_hist[i] = 0;
  __syncthreads();
  const uint64_t E = prefix[nf];
  for (uint64_t chunk = blockIdx.x; chunk * kEpb < E; chunk += gridDim.x) {
    const uint64_t e0 = chunk * kEpb;
    const uint64_t e1 = (e0 + kEpb < E) ? e0 + kEpb : E;
    const int cnt = stage_chunk(chunk, chunk_rows, queue, prefix, offsets, cr);
    walk_strided(e0, e1, cnt, cr, cols, [&](uint32_t w, uint32_t) { atomicAdd(&s_hist[w >> shift], 1u); });
    __syncthreads();
  }
  for (int i = threadIdx.x; i < nb; i += kBlock)
    if (s_hist[i]) atomicAdd(bucket_cnt + i, (unsigned long long)s_hist[i]);
}

// bucket_cnt -> exclusive offsets in bucket_cur (one block; nb <= kBinMaxBuckets)
__global__ void __launch_bounds__(kBlock) k_td_bin_offsets(const unsigned long long* __restrict__ bucket_cnt,
                                                           int nb, unsigned long long* __restrict__ bucket_cur) {
  if (threadIdx.x == 0) {
    unsigned long long run = 0;
    for (int i = 0; i < nb; ++i) {
      bucket_cur[i] = run;
      run += bucket_cnt[i];
    }
  }
}

__global__ void __launch_bounds__(kBlock) k_td_bin_scatter(const uint32_t* __restrict__ queue, int64_t nf,
                                                           const uint64_t* __restrict__ prefix,
                                                           const uint32_t* __restrict__ chunk_rows,
                                                           const uint64_t* __restrict__ offsets,
                                                           const uint32_t* __restrict__ cols, int shift, int nb,
                                                           unsigned long long* __restrict__ bucket_cur,
                                                           uint64_t* __restrict__ pairs) {
  __shared__ ChunkRows cr;
  __shared__ unsigned long long s_cur[kBinMaxBuckets];
  __shared__ unsigned s_hist[kBinMaxBuckets];
  const uint64_t E = prefix[nf];
  for (uint64_t chunk = blockIdx.x; chunk * kEpb < E; chunk += gridDim.x) {
    const uint64_t e0 = chunk * kEpb;
    const uint64_t e1 = (e0 + kEpb < E) ? e0 + kEpb : E;
    for (int i = threadIdx.x; i < nb; i += kBlock) s_hist[i] = 0;
    const int cnt = stage_chunk(chunk, chunk_rows, queue, prefix, offsets, cr);  // ends with a barrier
    walk_strided(e0, e1, cnt, cr, cols, [&](uint32_t w, uint32_t) { atomicAdd(&s_hist[w >> shift], 1u); });
    __syncthreads();
    for (int i = threadIdx.x; i < nb; i += kBlock)
      s_cur[i] = s_hist[i] ? atomicAdd(bucket_cur + i, (unsigned long long)s_hist[i]) : 0;
    __syncthreads();
    walk_strided(e0, e1, cnt, cr, cols, [&](uint32_t w, uint32_t u) {
      const unsigned long long pos = atomicAdd(&s_cur[w >> shift], 1ull);
      pairs[pos] = ((uint64_t)w << 32) | u;
    });
    __syncthreads();
  }
}

// Applies the pairs in order.  The grid strides over them together, so the
// pairs in flight at any moment span a window of grid * kBlock pairs, i.e.
// one or two target ranges, whose level and parent lines stay in L2.
__global__ void __launch_bounds__(kBlock) k_td_bin_apply(const uint64_t* __restrict__ pairs, uint64_t E,
                                                         uint8_t* level, uint32_t* __restrict__ parent,
                                                         uint32_t lvl) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < E; i += stride) {
    const uint64_t x = pairs[i];
    const uint32_t w = (uint32_t)(x >> 32);
    if (level[w] != 0xFF) continue;
    level[w] = (uint8_t)lvl;
    parent[w] = (uint32_t)x;
  }
}

// After a bulk top-down level: the vertices whose level became 'lvl' join the
// visited bitmap and form the frontier bitmap; their number goes to counters.
// A wave takes 16 bitmap words (1024 vertices) per step: lane i reads 16
// level bytes with one 16-byte load (1 KiB per wave instruction), and lanes
// 4k..4k+3 assemble word k with two shuffles.
__device__ __forceinline__ uint32_t bytes_equal4(uint32_t x, uint32_t pat) {
  const uint32_t y = x ^ pat;
  uint32_t r = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) r |= (((y >> (8 * b)) & 0xFFu) == 0 ? 1u : 0u) << b;
  return r;
}

__global__ void __launch_bounds__(kBlock) k_td_finish(const uint8_t* __restrict__ level, int64_t rows,
                                                      int64_t words, uint32_t lvl, uint64_t* __restrict__ vis,
                                                      uint64_t* __restrict__ fbits,
                                                      unsigned long long* __restrict__ counters,
                                                      const uint64_t* __restrict__ prefix, int64_t nf) {
  if (prefix[nf] <= kTdSmall) return;  // a small level: k_td_expand<false> kept the queue exact
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (kBlock / 64);
  const int64_t groups = (words + 15) / 16;
  const uint32_t pat = (lvl & 0xFFu) * 0x01010101u;
  uint64_t total = 0;
  for (int64_t gi = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); gi < groups; gi += nwaves) {
    const int64_t v0 = gi * 1024 + lane * 16;
    uint32_t m16 = 0;
    if (v0 + 16 <= rows) {
      const uint4 q = *reinterpret_cast<const uint4*>(level + v0);  // v0 is a multiple of 16
      m16 = bytes_equal4(q.x, pat) | (bytes_equal4(q.y, pat) << 4) | (bytes_equal4(q.z, pat) << 8) |
            (bytes_equal4(q.w, pat) << 12);
    } else {
      for (int j = 0; j < 16; ++j)
        if (v0 + j < rows && level[v0 + j] == (uint8_t)lvl) m16 |= 1u << j;
    }
    uint64_t m = (uint64_t)m16 << (16 * (lane & 3));
    m |= __shfl_xor(m, 1, 64);
    m |= __shfl_xor(m, 2, 64);
    const int64_t w = gi * 16 + (lane >> 2);
    if ((lane & 3) == 0 && w < words) {
      vis[w] |= m;
      fbits[w] = m;
      total += __popcll(m);
    }
  }
  block_add(total, stripe_of(counters + kStripeBase, S_FOUND));
}

// Frontier bitmap -> frontier queue in ascending vertex order: an exclusive
// scan of per-word popcounts gives every word its output position, so no
// atomics are involved.  The bits are 'now & ~before' (before may be null).
struct FrontierBits {
  const uint64_t* now;
  const uint64_t* before;
  __device__ uint64_t operator()(size_t w) const {
    const uint64_t x = before ? (now[w] & ~before[w]) : now[w];
    return (uint64_t)__popcll(x);
  }
};
struct FrontierEmit {
  const uint64_t* now;
  const uint64_t* before;
  uint32_t* queue;
  __device__ void operator()(size_t w, uint64_t pre) const {
    uint64_t x = before ? (now[w] & ~before[w]) : now[w];
    while (x) {
      queue[pre++] = (uint32_t)(w * 64 + __builtin_ctzll(x));
      x &= x - 1;
    }
  }
};

// --- algorithmic byte model, evaluated from the final levels -------------
// top-down level L reads the rows of the vertices at level L-1
__global__ void __launch_bounds__(kBlock) k_model_td(const uint8_t* __restrict__ level,
                                                     const uint64_t* __restrict__ offsets, int64_t rows,
                                                     uint32_t L, unsigned long long* acc) {
  uint64_t b = 0;
  for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < rows; v += (int64_t)gridDim.x * kBlock)
    if (level[v] == L - 1) b += 12 + 4 * (offsets[v + 1] - offsets[v]);
  block_add(b, acc);
}

// bottom-up level L probes, for every vertex with edges still unvisited, its
// neighbours in ascending order up to the first one visited before L
__global__ void __launch_bounds__(kBlock) k_model_bu(const uint8_t* __restrict__ level,
                                                     const uint64_t* __restrict__ offsets,
                                                     const uint32_t* __restrict__ cols, int64_t rows,
                                                     uint32_t L, unsigned long long* acc) {
  uint64_t b = 0;
  for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < rows; v += (int64_t)gridDim.x * kBlock) {
    const uint8_t lv = level[v];
    if (lv != 0xFF && lv < L) continue;
    const uint64_t s = offsets[v], e = offsets[v + 1];
    if (s == e) continue;
    uint64_t k = 0;
    for (uint64_t j = s; j < e; ++j) {
      ++k;
      const uint8_t lw = level[cols[j]];
      if (lw != 0xFF && lw < L) break;
    }
    b += 8 + 4 * k;
  }
  block_add(b, acc);
}

void bfs_model_bytes(g5_ctx* ctx, double* per_level, double* total) {
  Graph& g = ctx->graph;
  BfsState& b = ctx->bfs;
  G5_CHECK(b.have_result, "g5_bfs_model_bytes: no BFS result (call g5_run_bfs first)");
  const g5_bfs_stats& st = b.stats;
  hipStream_t s = ctx->stream;
  ctx->acc.alloc(4);
  const int64_t rows = g.n_rows;
  double tot = 1.0;  // the root's level byte
  for (int L = 0; L < G5_MAX_LEVELS; ++L)
    if (per_level) per_level[L] = 0;
  for (int L = 1; L < st.num_levels; ++L) {
    G5_HIP(hipMemsetAsync(ctx->acc.p, 0, 8, s));
    const unsigned grid = grid_of(rows, kBlock, 8192);
    if (st.direction[L])
      hipLaunchKernelGGL(k_model_td, dim3(grid), dim3(kBlock), 0, s, b.level.p, g.offsets.p, rows,
                         (uint32_t)L, (unsigned long long*)ctx->acc.p);
    else
      hipLaunchKernelGGL(k_model_bu, dim3(grid), dim3(kBlock), 0, s, b.level.p, g.offsets.p, g.cols.p,
                         rows, (uint32_t)L, (unsigned long long*)ctx->acc.p);
    G5_HIP(hipGetLastError());
    uint64_t h = 0;
    G5_HIP(hipMemcpyAsync(&h, ctx->acc.p, 8, hipMemcpyDeviceToHost, s));
    G5_HIP(hipStreamSynchronize(s));
    const double nq = (double)st.nq[L];
    double bytes = (double)h + nq;  // + 1 B level write per discovered vertex
    if (st.direction[L]) bytes += 4.0 * nq;             // queue write
    else bytes += 3.0 * (double)g.n / 8.0;              // visited read, next read+write
    if (per_level) per_level[L] = bytes;
    tot += bytes;
  }
  if (total) *total = tot;
}

__global__ void k_make_pred(const uint32_t* __restrict__ old2new, const uint32_t* __restrict__ new2old,
                            const uint8_t* __restrict__ level, const uint32_t* __restrict__ parent,
                            int64_t n, int64_t rows, int64_t root_orig, int64_t* __restrict__ pred) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t nv = old2new[v];
    int64_t out = -1;
    if (v == root_orig) {
      out = root_orig;
    } else if ((int64_t)nv < rows) {
      const uint8_t l = level[nv];
      if (l != 0xFF) out = (int64_t)new2old[parent[nv]] | ((int64_t)l << 48);
    }
    pred[v] = out;
  }
}

__global__ void __launch_bounds__(kBlock) k_make_levels(const uint32_t* __restrict__ old2new,
                                                        const uint8_t* __restrict__ level, int64_t n, int64_t rows,
                                                        int64_t root_orig, uint8_t* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q * 16 < n; q += stride) {
    const int m = n < 16 ? (int)n : 16;  // n is a power of two
    alignas(16) uint32_t nv[16];
    if (m == 16) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        reinterpret_cast<uint4*>(nv)[j] = reinterpret_cast<const uint4*>(old2new + q * 16)[j];
    } else {
      for (int j = 0; j < 16; ++j) nv[j] = j < m ? old2new[j] : 0xFFFFFFFFu;
    }
    uint32_t l[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) l[j] = j < m && (int64_t)nv[j] < rows ? level[nv[j]] : 0xFF;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = l[4 * j] | (l[4 * j + 1] << 8) | (l[4 * j + 2] << 16) | (l[4 * j + 3] << 24);
    const int64_t r = root_orig - q * 16;  // also a root without edges, which is no row of the CSR
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (r >= 4 * j && r < 4 * j + 4) w[j] &= ~(0xFFu << (8 * (r & 3)));
    if (m == 16) {
      reinterpret_cast<uint4*>(out)[q] = uint4{w[0], w[1], w[2], w[3]};
    } else {
      for (int j = 0; j < m; ++j) out[j] = (uint8_t)(w[j >> 2] >> (8 * (j & 3)));
    }
  }
}

void launch_make_levels(const uint32_t* old2new, const uint8_t* row_level, int64_t n, int64_t rows, int64_t root,
                        uint8_t* out, hipStream_t s) {
  hipLaunchKernelGGL(k_make_levels, dim3(grid_of((n + 15) / 16, kBlock, 4096)), dim3(kBlock), 0, s, old2new, row_level,
                     n, rows, root, out);
  G5_HIP(hipGetLastError());
}

// Tuple weights of the reached rows: 16 rows per thread and turn, one sum per
// workgroup published to the host, which adds them up (at most kTepsGrid).
// Bound by the 5 B read per row: 141 us at S28, 290 with adds to one word and
// a copy of the sum.
constexpr int kTepsGrid = 256;
constexpr int kTepsThreads = 1024;
__global__ void __launch_bounds__(kTepsThreads) k_teps(const uint8_t* __restrict__ level,
                                                       const uint32_t* __restrict__ weight, int64_t rows,
                                                       Published* pub, uint64_t seq) {
  __shared__ uint64_t s_sum[kTepsThreads / 64];
  uint64_t sum = 0;
  const int64_t stride = (int64_t)gridDim.x * kTepsThreads;
  for (int64_t q = (int64_t)blockIdx.x * kTepsThreads + threadIdx.x; q * 16 < rows; q += stride) {
    if (q * 16 + 16 <= rows) {
      alignas(16) uint32_t l[4];
      *reinterpret_cast<uint4*>(l) = reinterpret_cast<const uint4*>(level)[q];
      uint4 w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = reinterpret_cast<const uint4*>(weight)[q * 4 + j];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sum += (l[j] & 0xFF) != 0xFF ? w[j].x : 0;
        sum += ((l[j] >> 8) & 0xFF) != 0xFF ? w[j].y : 0;
        sum += ((l[j] >> 16) & 0xFF) != 0xFF ? w[j].z : 0;
        sum += (l[j] >> 24) != 0xFF ? w[j].w : 0;
      }
    } else {
      for (int64_t v = q * 16; v < rows; ++v) sum += level[v] != 0xFF ? weight[v] : 0;
    }
  }
  sum = wave_sum(sum);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x < 64) {
    const uint64_t t = wave_sum(threadIdx.x < kTepsThreads / 64 ? s_sum[threadIdx.x] : 0);
    if (threadIdx.x == 0) publish(pub + blockIdx.x, t, seq);
  }
}

// --- steps: the levels a search decides for itself -----------------------------
// A search is an init launch and a row of step launches, each of which starts
// by folding the previous step's vertex count into the search's state and
// applying the reference's switch rule (mpi/bfs.hpp:2799-2829), so that a
// level costs one launch and no host round trip (18 us a level before, of 4 to
// 12 us of kernel on graphs up to SCALE 21).  Every workgroup folds the same
// values and so takes the same decision; workgroup 0 passes the state on.
// The host keeps one step queued behind the running one until a step
// publishes the end; steps launched past it find it and leave.  A step runs
//   * consecutive small top-down levels (at most kStepNf vertices with at
//     most small_edges edges each) in workgroup 0 alone;
//   * a top-down level of at most kTdSmall edges: every workgroup makes the
//     frontier's degree prefix in LDS, the waves take 256 edges at a time (row
//     by binary search in LDS), test-and-set the visited bitmap and append
//     the winners through an LDS list;
//   * a bottom-up level: a wave reads `span` bitmap words at a time (one
//     coalesced load, one word per lane) and probes those with an unvisited
//     vertex (step_bottom_up); late levels, where almost every word is full,
//     cost little more than a pass over the bitmap.  The new vertices are listed as well, as far as
//     each workgroup's LDS list holds them, for a top-down level that follows;
// and hands any other level back to the host (larger top-down levels, a
// frontier whose queue has to be rebuilt from the bitmaps).  Graphs of one
// workgroup's size run all their levels in one step.
constexpr int kStepThreads = 1024;
constexpr int kStepNf = 4096;
constexpr int kBuWords = 4;        // open words whose first probes are in flight together (bottom-up)
constexpr int kBuSpan = 16;        // most words of a bottom-up turn
constexpr int kStepList = 2048;    // LDS list of a workgroup's new vertices
constexpr int kStepMaxGrid = 256;  // most workgroups of a step: kTdSmall edges are 4,096 waves of 256
constexpr int kStepMaxLevel = 254; // levels are bytes, 0xFF = unreached
enum { STEP_GO = 0, STEP_DONE = 1, STEP_LARGE = 2, STEP_QUEUE = 3, STEP_LIMIT = 4, STEP_BOTTOM_UP = 5 };

struct StepState {
  int32_t lvl;       // levels completed
  int32_t stop;
  int32_t forward, growing;
  int32_t cur, qi;   // current visited bitmap, queue holding the frontier
  int32_t queued;    // queue[qi] holds the frontier whole
  int32_t pending;   // 1: a level has run whose count is still in the counters, 2: by the bottom-up body
  int64_t nf;        // frontier of the coming level
  int64_t prev_nq, visited;
  uint64_t edges;    // its edges, where a step that hands the level back has summed them (0: not known)
  uint64_t start;    // clock at the start of the pending level
};

// Control words: three sets of {queue count, list overflow, found stripes} in
// turn by step (a step adds to its own, reads the previous one's and clears
// the next one's), the passed state (two slots in turn), the clock of the start.
constexpr int kSetWords = 2 * kStripeWords + kStripes * kStripeWords;
enum { SET_QUEUE = 0, SET_OVER = kStripeWords, SET_FOUND = 2 * kStripeWords };
constexpr int kStateWords = 16;
static_assert(sizeof(StepState) <= kStateWords * 8, "state slot");
constexpr int kStepState = 3 * kSetWords;
constexpr int kStepClock = kStepState + 2 * kStateWords;
constexpr int kStepArgs = kStepClock + 8;  // the arguments every step reads (StepArgs)
constexpr int kStepWords = kStepArgs + 32;

// Published: two entries per level (count, kind and clock ticks), then
enum { P_STEP = 2 * (kStepMaxLevel + 1), P_STOP, P_LVL, P_BITS, P_NF, P_PREV, P_VISITED, P_EDGES, P_TICKS, P_NUM };

struct StepArgs {
  const uint64_t* offsets;
  const uint32_t* cols;
  const uint32_t* first_nbr;
  uint64_t* vis[2];
  uint32_t* queue[3];
  uint8_t* level;
  uint32_t* parent;
  Published* pub;
  int64_t words, n_active, small_edges, tail_pull;
  int span;   // words per wave turn of a bottom-up level
  int share;  // its rows are shared out in the workgroup
  int host_bu;  // bottom-up levels go back to the host
};

__device__ __forceinline__ void step_publish_level(const StepArgs& a, uint64_t seq, int lvl, int64_t nq, int kind,
                                                   uint64_t ticks) {
  publish(a.pub + 2 * lvl, ((uint64_t)nq << 2) | (uint64_t)kind, seq);
  publish(a.pub + 2 * lvl + 1, ticks, seq);
}

// Least workgroups of a step, the bitmap words and edges up to which one
// workgroup takes the whole search in one launch (S10, 14 words: 47 us a
// search, 48 in steps of many; S12, 53 words: its large level takes 38 us
// alone and 13 in 64 workgroups), the bitmap words beyond
// which bottom-up levels go back to the host, and the steps launched ahead.
constexpr unsigned kStepMinGrid = 64;
static_assert(kStepMinGrid <= (unsigned)kStepMaxGrid, "workgroups of a step");
constexpr int64_t kStepAloneWords = 32;
constexpr int64_t kStepShareWords = 8192;  // see step_bottom_up
constexpr int64_t kStepAloneEdges = 1 << 18;
constexpr int64_t kStepMaxWords = 100000;
constexpr int kStepAhead = 3;

// Counts a finished level in (kind: bit 0 forward, bit 1 bottom-up body) and
// applies the switch rule.
__host__ __device__ __forceinline__ void step_fold(int64_t n_active, StepState& st, int64_t nq) {
  ++st.lvl;
  st.visited += nq;
  st.nf = nq;
  if (nq == 0) {
    st.stop = STEP_DONE;
    return;
  }
  const double na = (double)n_active;
  if (st.growing && nq > st.prev_nq) {
    if (st.forward && (double)nq > na / 2000.0) st.forward = 0;
  } else if (!st.forward && n_active - st.visited < (int64_t)(na / 8.0)) {
    st.forward = 1;
    st.growing = 0;
  }
  st.prev_nq = nq;
}

// A top-down level after the bottom-up phase whose frontier holds more than
// 1/tail_pull as many vertices as remain unvisited (and more than kStepNf) is
// found by the bottom-up body: an unvisited vertex with a visited neighbour is
// on this level (an older neighbour would have reached it before), so both
// find the same vertices, and this one probes from the few unvisited ones
// instead of expanding the frontier.  The level keeps its top-down place in
// the schedule.
__host__ __device__ __forceinline__ bool tail_pulls(int forward, int growing, int64_t tail_pull, int64_t nf,
                                                    int64_t unvisited) {
  return forward && !growing && tail_pull > 0 && nf > kStepNf && tail_pull * nf > unvisited;
}

static_assert(sizeof(StepArgs) <= 32 * 8, "argument block");

// What a workgroup of kWaves waves keeps of a bottom-up turn.
template <int kWaves>
struct BuLds {
  uint16_t miss[kWaves * kBuSpan * 64];
  uint32_t got[kWaves * kBuSpan * 2];
  uint32_t n[kWaves];
};

struct StepLds {
  union {
    uint64_t base[kStepNf];  // cols index of frontier row i's first entry - pre[i]
    BuLds<kStepThreads / 64> bu;
  };
  uint32_t pre[kStepNf + 1];  // first virtual edge of the row
  uint32_t src[kStepNf];
  uint32_t list[kStepList];
  uint64_t wave[kStepThreads / 64];
  uint32_t n;
  uint64_t lap;  // clock at the start of a level of workgroup 0's own
  union {
    StepState st;
    uint64_t st_words[kStateWords];
  };
};

// Degree prefix of the frontier in LDS (cur[0, nf), nf <= kStepNf); returns
// its edge count.  The 32-bit prefix is whole when that is at most 2^32 - 1.
__device__ __forceinline__ uint64_t step_prefix(StepLds& L, const uint32_t* __restrict__ cur, int nf,
                                                const uint64_t* __restrict__ offsets) {
  constexpr int kPer = kStepNf / kStepThreads;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int per = (nf + kStepThreads - 1) / kStepThreads;  // entries per thread
  uint64_t o[kPer], d[kPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = t * per + j;
    o[j] = d[j] = 0;
    if (j < per && i < nf) {
      const uint32_t u = cur[i];
      L.src[i] = u;
      o[j] = offsets[u];
      d[j] = offsets[u + 1] - o[j];
    }
    sum += d[j];
  }
  const uint64_t inc = wave_incl_scan(sum);
  if (lane == 63) L.wave[wave] = inc;
  if (t == 0) L.n = 0;
  __syncthreads();
  uint64_t run = inc - sum, total = 0;
  for (int w = 0; w < kStepThreads / 64; ++w) {
    if (w < wave) run += L.wave[w];
    total += L.wave[w];
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = t * per + j;
    if (j < per && i < nf) {
      L.pre[i] = (uint32_t)run;
      L.base[i] = o[j] - run;
    }
    run += d[j];
  }
  __syncthreads();
  return total;
}

// Row of virtual edge e: the last one that starts at or before it.
__device__ __forceinline__ int step_row(const StepLds& L, int nf, uint32_t e) {
  int lo = 0, hi = nf - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (L.pre[mid] <= e) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Sets bit w of the bitmap for every lane with ok; true for the one lane whose
// claim finds it unset.  Every lane of the wave calls it.  Neighbouring lanes
// whose targets share a word (a row is sorted, and every row holds the hubs)
// claim with one atomic: the frontier's rows all meet in the first words, and
// atomics on one word are performed one after another (160 rows, 10,000 claims
// of the hubs' words: 0.18 ms of a level of 0.05 at SCALE 23).
__device__ __forceinline__ bool claim_bits(uint64_t* vis, uint32_t w, bool ok) {
  const int lane = threadIdx.x & 63;
  const uint32_t key = ok ? w >> 6 : 0x80000000u | (uint32_t)lane;  // words are below 2^26
  const uint64_t bit = ok ? UINT64_C(1) << (w & 63) : 0;
  const uint32_t left = __shfl_up(key, 1, 64);
  const uint64_t heads = __ballot(lane == 0 || key != left);  // first lanes of the runs
  const uint64_t upto = ~UINT64_C(0) >> (63 - lane);
  const int start = 63 - __builtin_clzll(heads & upto);
  const uint64_t later = heads & ~upto;
  const int end = later ? __builtin_ctzll(later) - 1 : 63;
  uint64_t run = bit;  // OR over the run up to this lane
  if (heads != ~UINT64_C(0)) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t x = __shfl_up(run, o, 64);
      if (lane - o >= start) run |= x;
    }
  }
  uint64_t before = __shfl_up(run, 1, 64);
  if (lane == start) before = 0;
  uint64_t old = 0;
  if (ok && lane == end) old = atomicOr((unsigned long long*)(vis + key), (unsigned long long)run);
  old = __shfl(old, end, 64);
  return ok && !((old | before) & bit);
}

// A lane's claims of the edges e, e + stride, ... below end, four in flight:
// rows, columns and the bitmap filter of all four before the first claim.
// Every lane of the wave calls it.
template <class F>
__device__ __forceinline__ void step_expand(const StepArgs& a, const StepLds& L, int nf, uint64_t* vis, uint32_t e,
                                            uint32_t end, uint32_t stride, int lvl, F&& append) {
  uint32_t w[4], u[4];
  bool ok[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t x = e + j * stride;
    ok[j] = x < end;
    w[j] = u[j] = 0;
    if (ok[j]) {
      const int i = step_row(L, nf, x);
      u[j] = L.src[i];
      w[j] = a.cols[L.base[i] + x];
    }
  }
  uint64_t b[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) b[j] = ok[j] ? vis[w[j] >> 6] : 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) ok[j] = claim_bits(vis, w[j], ok[j] && !((b[j] >> (w[j] & 63)) & 1));
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (ok[j]) {
      a.level[w[j]] = (uint8_t)lvl;
      a.parent[w[j]] = u[j];
      append(w[j]);
    }
}

// The bottom-up body.  A wave of the workgroup takes `span` words a turn,
// probes the first neighbours of kBuWords open words at a time and lists who
// missed; the rows of those are then searched with every lane busy, whatever
// words they come from (got gathers who was found).  Searched word by word, a
// turn of 128 vertices waited for six dependent loads (searches, us: S14 85,
// now 67; S21 131, 119; S24 318, 302; S28 2,560, 2,475; with the rows by groups
// 294 and 2,224, where k_bu's largest level moves 1 GB in 500 us).  `share`: the
// workgroup's waves share the rows out, so that a word of hubs, whose long
// rows one wave searches one after another, does not hold the level up;
// where waves have words enough that costs more than it gives (S14 18 -> 13
// us a level, S23 36 -> 40).  With a list (LDS, kStepList entries and their
// count) found vertices are appended to it.  Every thread of the workgroup
// calls it.  kSpread: neighbouring turns go to different workgroups (hubs are
// neighbours).  Returns the lane's share of the count.
template <int kWaves, int kU, int kR, bool kSpread>
__device__ __forceinline__ uint64_t step_bottom_up(const StepArgs& a, BuLds<kWaves>& B, uint32_t* list,
                                                   uint32_t* list_n, const uint64_t* __restrict__ vis,
                                                   uint64_t* __restrict__ vis_next, int lvl, bool share) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, span = a.span;
  const uint64_t below = lane ? ~UINT64_C(0) >> (64 - lane) : 0;
  // list position of the first of n new vertices (a full list stays full: further counts are not needed)
  const auto list_at = [&](uint32_t n) {
    uint32_t pos = kStepList;
    if (lane == 0 && n && *list_n <= (uint32_t)kStepList) pos = atomicAdd(list_n, n);
    return (uint32_t)__builtin_amdgcn_readfirstlane(pos);
  };
  const auto found = [&](int64_t v, uint32_t p, uint32_t pos) {
    a.level[v] = (uint8_t)lvl;
    a.parent[v] = p;
    if (list && pos < (uint32_t)kStepList) list[pos] = (uint32_t)v;
  };
  uint64_t total = 0;
  // word j of wave w's turn has slot w * kBuSpan + j
  const auto word_of = [&](int64_t turn, int slot) {
    const int w = slot / kBuSpan;
    const int64_t at = kSpread ? (turn * kWaves + w) * gridDim.x + blockIdx.x
                               : (turn * gridDim.x + blockIdx.x) * kWaves + w;
    return at * span + slot % kBuSpan;
  };
  uint32_t* got = B.got + wave * kBuSpan * 2;
  uint32_t* count = share ? B.n : B.n + wave;
  uint16_t* miss = share ? B.miss : B.miss + wave * kBuSpan * 64;
  const int first = share ? wave : 0, step = share ? kWaves : 1;
  const auto sync = [&] {
    if (share) __syncthreads();
    else wave_sync();
  };
  for (int64_t turn = 0; turn * kWaves * gridDim.x * span < a.words; ++turn) {
    const int64_t base = word_of(turn, wave * kBuSpan), wl = base + lane;
    const bool mine = lane < span && wl < a.words;
    const uint64_t cl = mine ? vis[wl] : ~UINT64_C(0);  // lanes beyond the span or the end read as visited
    if (lane < 2 * span) got[lane] = 0;
    if (share ? threadIdx.x == 0 : lane == 0) *count = 0;
    sync();
    for (uint64_t open = __ballot(cl != ~UINT64_C(0)); open;) {
      int j[kBuWords];
      uint32_t f[kBuWords];
      bool h[kBuWords];
      uint64_t m[kBuWords], r[kBuWords];
#pragma unroll
      for (int i = 0; i < kBuWords; ++i) {
        j[i] = open ? __builtin_ctzll(open) : -1;
        open &= open - 1;
        const uint64_t c = j[i] >= 0 ? __shfl(cl, j[i], 64) : ~UINT64_C(0);
        f[i] = (c >> lane) & 1 ? kNoNbr : a.first_nbr[(base + j[i]) * 64 + lane];
      }
#pragma unroll
      for (int i = 0; i < kBuWords; ++i) h[i] = f[i] != kNoNbr && bit_set(vis, f[i]);
      uint32_t pos = 0, out = 0;
#pragma unroll
      for (int i = 0; i < kBuWords; ++i) {
        m[i] = __ballot(h[i]);
        r[i] = __ballot(f[i] != kNoNbr && !h[i]);
        pos += (uint32_t)__popcll(m[i]);
        out += (uint32_t)__popcll(r[i]);
      }
      if (list) pos = list_at(pos);
      if (out) {
        if (lane == 0) out = atomicAdd(count, out);
        out = __builtin_amdgcn_readfirstlane(out);
      }
#pragma unroll
      for (int i = 0; i < kBuWords; ++i) {
        if (j[i] < 0) continue;
        if (lane < 2) got[2 * j[i] + lane] = (uint32_t)(m[i] >> (32 * lane));
        if (h[i]) found((base + j[i]) * 64 + lane, f[i], pos + (uint32_t)__popcll(m[i] & below));
        pos += (uint32_t)__popcll(m[i]);
        if ((r[i] >> lane) & 1)
          miss[out + (uint32_t)__popcll(r[i] & below)] = (uint16_t)((wave * kBuSpan + j[i]) * 64 + lane);
        out += (uint32_t)__popcll(r[i]);
      }
    }
    sync();
    const int nmiss = (int)*count;
    for (int i = first; i < nmiss; i += step * 64) {
      const bool in = i + lane * step < nmiss;
      const int x = in ? miss[i + lane * step] : 0;
      const int64_t v = word_of(turn, x >> 6) * 64 + (x & 63);
      uint32_t p = 0;
      const bool hit = row_marked_nbr<kU, kR>(in, (uint32_t)v, vis, a.offsets, a.cols, p);
      const uint64_t r = __ballot(hit);
      const uint32_t pos = list ? list_at((uint32_t)__popcll(r)) : 0;
      if (hit) {
        found(v, p, pos + (uint32_t)__popcll(r & below));
        atomicOr(B.got + (x >> 5), 1u << (x & 31));
      }
    }
    sync();
    if (mine) {
      const uint64_t n = got[2 * lane] | (uint64_t)got[2 * lane + 1] << 32;
      vis_next[wl] = cl | n;
      total += __popcll(n);
    }
  }
  return total;
}

// The address of the argument block, opaque from here on: fields are loaded
// where they are used instead of being held in registers across the bodies.
__device__ __forceinline__ const StepArgs& step_args(const unsigned long long* ctl) {
  const StepArgs* p = reinterpret_cast<const StepArgs*>(ctl + kStepArgs);
  asm volatile("" : "+s"(p));
  return *p;
}

__global__ void __launch_bounds__(kStepThreads) k_bfs_step(unsigned long long* __restrict__ ctl, int k, uint64_t seq) {
  __shared__ StepLds L;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const bool lead = blockIdx.x == 0;
  const uint64_t now = wall_clock64();
  // the state, with the previous step's level folded in (the same in every workgroup)
  if (wave == 0) {
    const unsigned long long* const set_prev = ctl + ((k + 2) % 3) * kSetWords;
    const uint64_t f = set_prev[SET_FOUND + lane * kStripeWords], over = set_prev[SET_OVER];
    if (lane < kStateWords) L.st_words[lane] = ctl[kStepState + ((k + 1) & 1) * kStateWords + lane];
    const int64_t nq = (int64_t)wave_sum(f);
    if (lane == 0) {
      const StepArgs& a = step_args(ctl);
      StepState& st = L.st;
      if (!st.stop && st.pending) {
        const bool bu = st.pending == 2;
        if (lead) step_publish_level(a, seq, st.lvl + 1, nq, st.forward | (st.pending & 2), now - st.start);
        st.queued = !bu || (nq <= kStepNf && !over);
        st.qi = st.qi == 2 ? 0 : st.qi + 1;
        if (bu) st.cur ^= 1;
        st.pending = 0;
        step_fold(a.n_active, st, nq);
      }
      if (!st.stop && st.nf == 0) st.stop = STEP_DONE;
      L.lap = now;
    }
  }
  if (lead) {
    unsigned long long* const set_next = ctl + ((k + 1) % 3) * kSetWords;
    for (int i = t; i < kSetWords; i += kStepThreads) set_next[i] = 0;
    if (t == 64) publish(step_args(ctl).pub + P_STEP, (uint64_t)k + 1, seq);
  }
  __syncthreads();
  const bool alone = gridDim.x == 1;
  // The queue the step starts from stays as it is while the step runs: every
  // workgroup makes its prefix, some after workgroup 0 has gone on to the next
  // small level.  Small levels use the other two in turn.
  const int entry = L.st.qi, lvl0 = L.st.lvl + 1;
  while (!L.st.stop) {
    const int lvl = __builtin_amdgcn_readfirstlane(L.st.lvl) + 1;
    int stop = STEP_GO;
    uint64_t E = 0;
    bool td = false;
    {
      const StepArgs& a = step_args(ctl);
      td = L.st.forward &&
           !tail_pulls(L.st.forward, L.st.growing, a.tail_pull, L.st.nf, a.n_active - L.st.visited);
      if (lvl > kStepMaxLevel) stop = STEP_LIMIT;
      else if (td && !L.st.queued) stop = STEP_QUEUE;
      else if (td && L.st.nf > kStepNf) stop = STEP_LARGE;
      else if (!td && a.host_bu) stop = STEP_BOTTOM_UP;
      if (!stop && td) {
        E = step_prefix(L, a.queue[L.st.qi], (int)L.st.nf, a.offsets);
        if (E > kTdSmall) stop = STEP_LARGE;
      }
    }
    if (stop) {
      __syncthreads();  // every thread has read L.st
      if (t == 0) {
        L.st.stop = stop;
        L.st.edges = E;
      }
      __syncthreads();
      break;
    }
    const int qi = __builtin_amdgcn_readfirstlane(L.st.qi);
    const int nqi = qi == entry ? (entry == 2 ? 0 : entry + 1) : 3 - entry - qi;
    unsigned long long* const set = ctl + (k % 3) * kSetWords;
    if (td) {
      const StepArgs& a = step_args(ctl);
      const bool small = alone || (int64_t)E <= a.small_edges;
      if (small && !lead) return;
      if (!small && lvl != lvl0) break;  // the other workgroups left at the first small level: the next step's
      const int nf = __builtin_amdgcn_readfirstlane((int)L.st.nf);
      uint64_t* const vis = a.vis[L.st.cur];
      uint32_t* const next = a.queue[nqi];
      if (small) {
        // the winners straight into the next queue
        for (uint32_t e = t; (e & ~63u) < (uint32_t)E; e += 4 * kStepThreads)  // whole waves
          step_expand(a, L, nf, vis, e, (uint32_t)E, kStepThreads, lvl,
                      [&](uint32_t w) { next[atomicAdd(&L.n, 1u)] = w; });
        __syncthreads();
        // the bitmap words the atomics changed are read past this CU's cache by a bottom-up level
        if (alone) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (t == 0) {
          const uint32_t n = L.n;
          const uint64_t end = wall_clock64();
          step_publish_level(a, seq, lvl, (int64_t)n, L.st.forward, end - L.lap);
          L.lap = end;
          L.st.qi = nqi;
          L.st.queued = 1;
          step_fold(a.n_active, L.st, (int64_t)n);
        }
        __syncthreads();
        if (!alone && (!L.st.forward || tail_pulls(L.st.forward, L.st.growing, a.tail_pull, L.st.nf,
                                                   a.n_active - L.st.visited)))
          break;  // a bottom-up level takes the grid
        continue;
      }
      // consecutive stretches go to different workgroups, so that the winners
      // spread over their lists (past a full list each costs a global atomic)
      const uint32_t nblk = gridDim.x;
      for (uint32_t c = wave * nblk + blockIdx.x; (uint64_t)c * 256 < E; c += nblk * (kStepThreads / 64)) {
        const uint64_t end = (uint64_t)(c + 1) * 256 < E ? (uint64_t)(c + 1) * 256 : E;
        step_expand(a, L, nf, vis, c * 256 + lane, (uint32_t)end, 64, lvl, [&](uint32_t w) {
          const uint32_t pos = atomicAdd(&L.n, 1u);
          if (pos < (uint32_t)kStepList) L.list[pos] = w;
          else next[atomicAdd(set + SET_QUEUE, 1ull)] = w;
        });
      }
    } else {
      if (t == 0) L.n = 0;
      __syncthreads();
      const StepArgs& a = step_args(ctl);
      const int cur = __builtin_amdgcn_readfirstlane(L.st.cur);
      const uint64_t f = wave_sum(step_bottom_up<kStepThreads / 64, 8, 4, true>(a, L.bu, L.list, &L.n, a.vis[cur],
                                                                          a.vis[cur ^ 1], lvl,
                                                                          a.share));
      if (lane == 0) L.wave[wave] = f;
    }
    __syncthreads();
    // the level's vertices so far (a top-down level: all were listed or queued)
    const StepArgs& a = step_args(ctl);
    uint32_t* const next = a.queue[nqi];
    const uint32_t n = L.n;
    uint64_t found = 0;
    if (td) {
      found = n;
    } else {
      for (int w = 0; w < kStepThreads / 64; ++w) found += L.wave[w];
    }
    const bool whole = td || n <= (uint32_t)kStepList;  // a full list says nothing about the rest
    const uint32_t listed = !whole ? 0 : (n < (uint32_t)kStepList ? n : (uint32_t)kStepList);
    if (alone) {
      // a bottom-up level of the only workgroup
      for (uint32_t i = t; i < listed; i += kStepThreads) next[i] = L.list[i];
      __syncthreads();
      if (t == 0) {
        const uint64_t end = wall_clock64();
        step_publish_level(a, seq, lvl, (int64_t)found, L.st.forward | 2, end - L.lap);
        L.lap = end;
        L.st.qi = nqi;
        L.st.cur ^= 1;
        L.st.queued = whole;
        step_fold(a.n_active, L.st, (int64_t)found);
      }
      __syncthreads();
      continue;
    }
    // a level of the whole grid: the next step folds it
    __syncthreads();  // L.wave has been read
    if (t == 0) {
      if (found) atomicAdd(set + SET_FOUND + (blockIdx.x % kStripes) * kStripeWords, (unsigned long long)found);
      if (!whole) set[SET_OVER] = 1;
      L.wave[0] = listed ? atomicAdd(set + SET_QUEUE, (unsigned long long)listed) : 0;
      if (lead) {
        L.st.pending = td ? 1 : 2;
        L.st.start = L.lap;
      }
    }
    __syncthreads();
    const uint64_t at = L.wave[0];
    for (uint32_t i = t; i < listed; i += kStepThreads) next[at + i] = L.list[i];
    if (lead && t < kStateWords) ctl[kStepState + (k & 1) * kStateWords + t] = L.st_words[t];
    return;
  }
  // the end, a level for the host, or a level of the whole grid after small ones
  if (!lead) return;
  if (t < kStateWords) ctl[kStepState + (k & 1) * kStateWords + t] = L.st_words[t];
  if (L.st.stop && t >= 64 && t < 64 + 8) {
    const StepState& st = L.st;
    uint64_t v = 0;
    switch (t - 64 + P_STOP) {
      case P_STOP: v = (uint64_t)st.stop; break;
      case P_LVL: v = (uint64_t)st.lvl; break;
      case P_BITS:
        v = (uint64_t)(st.forward | (st.growing << 1) | (st.cur << 2) | (st.queued << 3) | (st.qi << 4));
        break;
      case P_NF: v = (uint64_t)st.nf; break;
      case P_PREV: v = (uint64_t)st.prev_nq; break;
      case P_VISITED: v = (uint64_t)st.visited; break;
      case P_EDGES: v = st.edges; break;
      default: v = wall_clock64() - ctl[kStepClock]; break;
    }
    publish(step_args(ctl).pub + P_STOP + (t - 64), v, seq);
  }
}

// A bottom-up level of a large graph, launched by the host: the body above in
// 256-thread workgroups without a list, at twice the waves per CU a step
// leaves room for (its registers and LDS hold 16).
__global__ void __launch_bounds__(kBlock) k_bu(StepArgs a, int cur, int lvl, unsigned long long* __restrict__ counters,
                                               uint64_t* __restrict__ stamp) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();  // the level starts
  __shared__ BuLds<kBlock / 64> bu;
  const uint64_t f = step_bottom_up<kBlock / 64, 4, 1, false>(a, bu, nullptr, nullptr, a.vis[cur], a.vis[cur ^ 1], lvl, false);
  block_add(f, stripe_of(counters + kStripeBase, S_FOUND));
}

// The state a row of steps goes on from after a level run by the host (slot:
// the one the next step reads).
__global__ void k_step_resume(unsigned long long* __restrict__ ctl, StepState st, int k) {
  *reinterpret_cast<StepState*>(ctl + kStepState + ((k + 1) & 1) * kStateWords) = st;
}

// Everything a search starts from: levels unreached, the visited bitmap (bits
// past the last row read as visited so no sweep ever picks them), the root on
// level 0 and in the queue, the control words and level counters zero.
__global__ void __launch_bounds__(kBlock) k_bfs_init(const uint32_t* __restrict__ old2new, int64_t root_orig,
                                                     int64_t rows, int64_t words, uint8_t* __restrict__ level,
                                                     uint32_t* __restrict__ parent, uint64_t* __restrict__ vis,
                                                     uint32_t* __restrict__ queue, unsigned long long* __restrict__ ctl,
                                                     unsigned long long* __restrict__ counters, StepArgs args,
                                                     int active) {
  const int64_t stride = (int64_t)gridDim.x * kBlock, me = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t r = old2new[root_orig];  // >= rows for a root without edges (modes 1 and 2)
  for (int64_t q = me; q * 16 < rows; q += stride) {
    if (q * 16 + 16 <= rows && (r < q * 16 || r >= q * 16 + 16)) {
      reinterpret_cast<uint4*>(level)[q] = uint4{~0u, ~0u, ~0u, ~0u};
    } else {
      for (int64_t v = q * 16; v < q * 16 + 16 && v < rows; ++v) level[v] = v == r ? 0 : 0xFF;
    }
  }
  for (int64_t w = me; w < words; w += stride) {
    const int64_t first = w * 64;
    uint64_t x = 0;
    if (first + 64 > rows) x = ~UINT64_C(0) << (rows - first);
    if (r < rows && (r >> 6) == w) x |= UINT64_C(1) << (r & 63);
    vis[w] = x;
  }
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < 3 * kSetWords; i += kBlock) ctl[i] = 0;
    for (int i = threadIdx.x; i < kBfsCounters; i += kBlock) counters[i] = 0;
    if (threadIdx.x == 0) {
      ctl[kStepClock] = wall_clock64();
      *reinterpret_cast<StepArgs*>(ctl + kStepArgs) = args;
      StepState st{};
      st.forward = st.growing = st.queued = 1;
      st.nf = active;  // a root without edges is the whole tree: the first step finds the end
      st.visited = 1;
      *reinterpret_cast<StepState*>(ctl + kStepState + kStateWords) = st;  // the slot step 0 reads
      if (r < rows) {
        parent[r] = (uint32_t)r;
        queue[0] = (uint32_t)r;
      }
    }
  }
}

__global__ void k_stamp(uint64_t* stamp) { *stamp = wall_clock64(); }  // a level starts

// Level end: the counters the host decides the next level with (and the
// level's frontier edge count after a top-down level) are published straight
// into coherent host memory, each tagged with the level's sequence number, so
// the host need not wait for a copy and a stream synchronisation; behind them
// the time since the level's stamp (an event on either side of a level took 7
// us of the stream).  One wave: lane i takes stripe i.
static_assert(kStripes == 64, "k_publish sums one stripe per lane of a wave");
__global__ void __launch_bounds__(64) k_publish(unsigned long long* __restrict__ counters,
                                                const uint64_t* __restrict__ prefix, int64_t nf, int forward,
                                                Published* pub, uint64_t seq,
                                                const uint64_t* __restrict__ stamp) {
  const int t = threadIdx.x;
  if (t == C_NUM) publish(pub + t, wall_clock64() - *stamp, seq);
  unsigned long long* mine = counters + kStripeBase + t * kStripeWords;
  const uint64_t found = wave_sum(mine[S_FOUND]);
  const uint64_t next_e = wave_sum(mine[S_NEXT_E]);
  // ready for the next level, with no fill launched before it
  mine[S_FOUND] = 0;
  mine[S_NEXT_E] = 0;
  if (t < C_NUM) {
    uint64_t v = (forward && t == C_AUX) ? prefix[nf] : (uint64_t)counters[t];
    if (t == C_FOUND) v += found;
    if (t == C_NEXT_E) v += next_e;
    counters[t] = 0;
    publish(pub + t, v, seq);
  }
}

// Waits for the level's counters (see PublishBlock::wait).
static void wait_published(BfsState& b, hipStream_t s) {
  b.pub.wait(0, C_NUM + 1, b.pub_seq, s, "g5_run_bfs: level counters were not published");
  for (int i = 0; i <= C_NUM; ++i) b.h_counters[i] = b.pub.value(i);
}

static void build_hub_index(g5_ctx* ctx, BfsState& b, hipStream_t s);

// Buffers of the segment-list levels, sized for the tuning so that no run
// allocates: a growing top-down level has at most n_active / 2000 frontier
// vertices (one more switches to bottom-up), so a head level's row suffixes
// take at most that many segments and a piece or block level that many
// times its pieces, within seg_max.  The block index of the first rows is
// built here too.  (The binned form, off by default, sizes its pair buffer
// by the level's edges inside the run.)
void bfs_tuning_buffers(g5_ctx* ctx) { bfs_tuning_buffers(ctx, ctx->bfs, ctx->stream); }

void bfs_tuning_buffers(g5_ctx* ctx, BfsState& b, hipStream_t s) {
  Graph& g = ctx->graph;
  if (b.hub_shift > 0 && b.hub_built_shift != b.hub_shift) build_hub_index(ctx, b, s);
  const int64_t seg_max = b.seg_max > 0 ? std::min<int64_t>(b.seg_max, kSegMax) : kSegMax;
  const int64_t nf_max = g.n_active / 2000 + 1;
  int64_t pieces = 1;
  if (b.td_pieces > 0) pieces = std::max<int64_t>(pieces, b.td_pieces);
  if (b.hub_shift > 0) pieces = std::max<int64_t>(pieces, b.hub_pieces);
  const size_t seg_n = (size_t)std::min<int64_t>(nf_max * pieces, seg_max) + 2;
  b.seg_pre.alloc(seg_n);
  b.seg_base.alloc(seg_n);
  b.seg_src.alloc(seg_n);
  b.seg_start.alloc(seg_n);
  b.seg_count.alloc(1);
  b.seg_scan_tmp.alloc(scan_tmp_elems(seg_n));
}

void bfs_prepare(g5_ctx* ctx) { bfs_prepare(ctx, ctx->bfs, ctx->stream); }

void bfs_prepare(g5_ctx* ctx, BfsState& b, hipStream_t s) {
  Graph& g = ctx->graph;
  G5_CHECK(g.built, "g5_prepare_bfs: no graph (call g5_construct first)");
  b.release();
  const int64_t rows = g.n_rows;
  b.words = (rows + 63) / 64;
  for (auto& v : b.vis) v.alloc(b.words);
  b.level.alloc(rows);
  b.parent.alloc(rows);
  for (auto& q : b.queue) q.alloc(rows);
  b.prefix.alloc(rows + 1);
  b.chunk_rows.alloc(2 * ((uint64_t)g.nnz / kEpb + 2));
  const size_t scan_n = (size_t)rows + 1;
  b.scan_tmp.alloc(scan_tmp_elems(scan_n));
  b.counters.alloc(kBfsCounters);
  bfs_tuning_buffers(ctx, b, s);
  static_assert(C_NUM < sizeof(b.h_counters) / 8, "host counters");
  G5_HIP(hipStreamSynchronize(s));  // the published blocks are reset below
  b.pub.alloc(C_NUM + 1);
  b.stamp.alloc(1);
  b.pub_seq = 0;
  b.step_ctl.alloc(kStepWords);
  b.step_pub.alloc(P_NUM);
  b.step_seq = 0;
  b.teps_pub.alloc(kTepsGrid);
  b.teps_seq = 0;
  if (!b.tick_khz) {
    int khz = 0;
    G5_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device));
    b.tick_khz = khz > 0 ? khz : 100000;
  }
  b.prepared = true;
}

// The block index of the first rows: as many as fit kHubIndexBytes.
constexpr int64_t kHubIndexBytes = INT64_C(512) << 20;

static void build_hub_index(g5_ctx* ctx, BfsState& b, hipStream_t s) {
  Graph& g = ctx->graph;
  const int shift = (int)b.hub_shift;
  const int64_t nb = ((g.n_rows - 1) >> shift) + 1;
  b.hub_pieces = nb + 1;
  b.hub_rows = std::min<int64_t>(g.n_rows, kHubIndexBytes / (4 * b.hub_pieces));
  b.hub_bnd.alloc((size_t)(b.hub_rows * b.hub_pieces));
  hipLaunchKernelGGL(k_hub_bounds, dim3(grid_of(b.hub_rows * b.hub_pieces, kBlock, 65536)), dim3(kBlock), 0,
                     s, g.offsets.p, g.cols.p, b.hub_rows, b.hub_pieces, shift, b.hub_bnd.p);
  G5_HIP(hipGetLastError());
  G5_HIP(hipStreamSynchronize(s));
  b.hub_built_shift = b.hub_shift;
}

void bfs_run(g5_ctx* ctx, int64_t root) { bfs_run(ctx, ctx->bfs, ctx->stream, root); }

// A top-down level too large for a step: the frontier's rows as one virtual
// edge list over the whole grid (see k_td_expand), then the switch rule.
static void large_top_down(g5_ctx* ctx, BfsState& b, hipStream_t s, StepState& state) {
  Graph& g = ctx->graph;
  const int64_t rows = g.n_rows, nf = state.nf, visited = state.visited;
  const int lvl = state.lvl + 1, cur = state.cur, qi = state.qi, qn = (qi + 1) % 3;
  const double na = (double)g.n_active;
  unsigned long long* cnt = (unsigned long long*)b.counters.p;
  g5_bfs_stats& st = b.stats;
  // the frontier's edges when the step or the level before summed them (-1:
  // not known, both forms are launched and the device picks)
  const int64_t e_next = state.edges ? (int64_t)state.edges : -1;
  hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, s, b.stamp.p);
  device_scan(FrontierDegree{b.queue[qi].p, g.offsets.p, nf}, StoreU64{b.prefix.p},
              (size_t)nf + 1, b.scan_tmp.p, s);
  if (b.bin_edges > 0) {
    // the binned form sizes its pair buffer from E: wait for it
    G5_HIP(hipMemcpyAsync(b.h_counters + 1, b.prefix.p + nf, 8, hipMemcpyDeviceToHost, s));
    G5_HIP(hipStreamSynchronize(s));
  }
  const uint64_t E_known = b.bin_edges > 0 ? b.h_counters[1] : 0;
  // past the bottom-up phase most targets are visited: a bulk level then
  // tests the visited bitmap before the level array
  const int probe_vis = (double)visited > na / 4 ? 1 : 0;
  // the level's frontier edge count when the previous level summed it
  const bool known_small = e_next >= 0 && (uint64_t)e_next <= kTdSmall;
  const bool known_bulk = e_next >= 0 && (uint64_t)e_next > kTdSmall;
  // while the search grows, a bulk level can take its rows block by
  // block (exact target blocks) or piece by piece (positional pieces)
  const int64_t seg_max = b.seg_max > 0 ? std::min<int64_t>(b.seg_max, kSegMax) : kSegMax;
  const bool blocked = b.hub_shift > 0 && !probe_vis && nf * b.hub_pieces <= seg_max;
  // a growing bulk level settles its highest-degree targets bottom-up
  // first (degree order only)
  bool head = b.td_head > 0 && !probe_vis && g.reorder_mode == 2;
  if (head && e_next > (int64_t)kTdSmall) {
    // E known on the host: no head when no row reaches the threshold
    // (the same test k_td_head_size makes)
    const double r = (double)g.nnz / (double)e_next;
    if ((double)b.td_head / 16.0 * r * r > (double)g.max_degree) head = false;
  }
  unsigned long long* head_words = head ? cnt + C_HEAD : nullptr;
  const bool pieces = blocked || (b.td_pieces > 0 && !probe_vis && nf * b.td_pieces <= seg_max);
  // with a head and row order, the expansion walks row suffixes (one
  // segment per frontier row: the segment count field bounds nf)
  if (head && !pieces && nf > seg_max) head = false;
  head_words = head ? cnt + C_HEAD : nullptr;
  const bool suffix = head && !pieces;
  const bool binned = b.bin_edges > 0 && E_known > kTdSmall && E_known >= (uint64_t)b.bin_edges;
  // Without binning no launch waits for E on the host: chunk rows and the
  // expansion take upper-bound grids and read E (prefix[nf]) on the
  // device; the small and the bulk expansion are both launched and the
  // one that does not fit E exits at once, as does k_td_finish after a
  // small level.  The host learns E with the level's counters.
  const uint64_t max_chunks = b.chunk_rows.n / 2;  // sized for every edge of the graph
  const uint64_t nchunks = b.bin_edges > 0 ? (E_known + kEpb - 1) / kEpb : max_chunks;
  const unsigned grid = b.bin_edges > 0 ? grid_of((int64_t)E_known, kEpb, 2048) : 2048u;
  if (nchunks)
    hipLaunchKernelGGL(k_chunk_rows<kEpb>,
                       dim3(b.bin_edges > 0 ? grid_of((int64_t)(2 * nchunks), kBlock, 65536) : 4096u),
                       dim3(kBlock), 0, s, b.prefix.p, nf, nchunks, b.chunk_rows.p);
  if (!known_bulk)
    hipLaunchKernelGGL(k_td_expand<false>, dim3(grid), dim3(kBlock), 0, s, b.queue[qi].p, nf, b.prefix.p,
                       b.chunk_rows.p, g.offsets.p, g.cols.p, b.vis[cur].p, b.level.p, b.parent.p,
                       b.queue[qn].p, cnt, (uint32_t)lvl, 0, nullptr);
  if (head && !binned && !known_small) {
    hipLaunchKernelGGL(k_td_head_size, dim3(1), dim3(1), 0, s, b.prefix.p, nf, g.offsets.p, rows, b.words,
                       (double)g.nnz, (double)b.td_head / 16.0, head_words);
    hipLaunchKernelGGL(k_td_head, dim3(grid_of(b.words, kBlock / 64, 8192)), dim3(kBlock), 0, s,
                       b.vis[cur].p, g.first_nbr.p, g.offsets.p, g.cols.p, b.level.p, b.parent.p, head_words,
                       (uint32_t)lvl);
    G5_HIP(hipGetLastError());
  }
  if (known_small) {
    // nothing else to launch: the small expansion keeps the queue exact
  } else if (binned) {
    // binned by target range (see k_td_bin_count)
    const uint64_t E = E_known;
    int shift = kBinShift;
    while ((rows >> shift) >= kBinMaxBuckets) ++shift;
    const int nb = (int)(((rows - 1) >> shift) + 1);
    b.bin_pairs.alloc(E);
    b.bin_cnt.alloc(2 * kBinMaxBuckets);
    unsigned long long* bc = (unsigned long long*)b.bin_cnt.p;
    G5_HIP(hipMemsetAsync(bc, 0, nb * 8, s));
    hipLaunchKernelGGL(k_td_bin_count, dim3(grid), dim3(kBlock), 0, s, b.queue[qi].p, nf, b.prefix.p,
                       b.chunk_rows.p, g.offsets.p, g.cols.p, shift, nb, bc);
    hipLaunchKernelGGL(k_td_bin_offsets, dim3(1), dim3(kBlock), 0, s, bc, nb, bc + kBinMaxBuckets);
    hipLaunchKernelGGL(k_td_bin_scatter, dim3(grid), dim3(kBlock), 0, s, b.queue[qi].p, nf, b.prefix.p,
                       b.chunk_rows.p, g.offsets.p, g.cols.p, shift, nb, bc + kBinMaxBuckets, b.bin_pairs.p);
    hipLaunchKernelGGL(k_td_bin_apply, dim3(grid_of((int64_t)E, kBlock, 2048)), dim3(kBlock), 0, s,
                       b.bin_pairs.p, E, b.level.p, b.parent.p, (uint32_t)lvl);
  } else if (pieces || suffix) {
    // segment-list bulk level; a small level makes an empty segment list
    // and the expansion exits (both read E on the device)
    const size_t np = (size_t)(suffix ? nf : nf * (blocked ? b.hub_pieces : b.td_pieces)) + 1;
    b.seg_pre.alloc(np);
    b.seg_base.alloc(np);
    b.seg_src.alloc(np);
    b.seg_count.alloc(1);
    b.seg_scan_tmp.alloc(scan_tmp_elems(np));
    if (suffix) {
      b.seg_start.alloc(np);
      hipLaunchKernelGGL(k_suffix_start, dim3(grid_of(nf, kBlock, 4096)), dim3(kBlock), 0, s, b.queue[qi].p, nf,
                         b.prefix.p, g.offsets.p, g.cols.p, head_words, b.seg_start.p);
      const SuffixLen sl{b.queue[qi].p, g.offsets.p, b.prefix.p, nf, 1, b.seg_start.p};
      device_scan(sl, PieceEmit<SuffixLen>{sl, b.seg_pre.p, b.seg_base.p, b.seg_src.p, b.seg_count.p}, np,
                  b.seg_scan_tmp.p, s);
    } else if (blocked) {
      const BlockLen bl{b.queue[qi].p, g.offsets.p, b.prefix.p, nf, b.hub_pieces, b.hub_bnd.p, b.hub_rows};
      device_scan(bl, PieceEmit<BlockLen>{bl, b.seg_pre.p, b.seg_base.p, b.seg_src.p, b.seg_count.p}, np,
                  b.seg_scan_tmp.p, s);
    } else {
      const PieceLen pl{b.queue[qi].p, g.offsets.p, b.prefix.p, nf, b.td_pieces};
      device_scan(pl, PieceEmit<PieceLen>{pl, b.seg_pre.p, b.seg_base.p, b.seg_src.p, b.seg_count.p}, np,
                  b.seg_scan_tmp.p, s);
    }
    hipLaunchKernelGGL(k_chunk_segs, dim3(4096), dim3(kBlock), 0, s, b.seg_pre.p, b.seg_count.p, max_chunks,
                       b.chunk_rows.p);
    hipLaunchKernelGGL(k_td_expand_segs, dim3(grid), dim3(kBlock), 0, s, b.prefix.p, nf, b.seg_pre.p,
                       b.seg_base.p, b.seg_src.p, b.seg_count.p, b.chunk_rows.p, g.cols.p, b.vis[cur].p,
                       b.level.p, b.parent.p, (uint32_t)lvl, head_words);
  } else {
    hipLaunchKernelGGL(k_td_expand<true>, dim3(grid), dim3(kBlock), 0, s, b.queue[qi].p, nf, b.prefix.p,
                       b.chunk_rows.p, g.offsets.p, g.cols.p, b.vis[cur].p, b.level.p, b.parent.p,
                       (uint32_t*)nullptr, cnt, (uint32_t)lvl, probe_vis, binned ? nullptr : head_words);
  }
  G5_HIP(hipGetLastError());
  // after a bulk level, k_td_finish makes vis[cur^1] exactly this level's
  // vertices and adds them to vis[cur]
  if (!known_small)
    hipLaunchKernelGGL(k_td_finish, dim3(grid_of((b.words + 15) / 16, kBlock / 64, 8192)), dim3(kBlock), 0,
                       s, b.level.p, rows, b.words, (uint32_t)lvl, b.vis[cur].p, b.vis[cur ^ 1].p, cnt,
                       b.prefix.p, nf);
  ++b.pub_seq;
  hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, s, cnt, b.prefix.p, nf, 1, b.pub.d, b.pub_seq,
                     b.stamp.p);
  G5_HIP(hipGetLastError());
  wait_published(b, s);
  const int64_t nq = (int64_t)b.h_counters[C_FOUND];
  const bool bulk = b.h_counters[C_AUX] > kTdSmall;
  st.direction[lvl] = 1;
  st.nq[lvl] = nq;
  st.num_levels = lvl + 1;
  st.level_ms[lvl] = (double)b.h_counters[C_NUM] / (double)b.tick_khz;
  ++state.lvl;
  state.visited += nq;
  state.nf = nq;
  state.edges = bulk ? 0 : b.h_counters[C_NEXT_E];  // a bulk level does not sum them
  if (nq == 0) return;
  // direction switch, mpi/bfs.hpp:2799-2829 (a top-down level hands over to bottom-up or goes on)
  if (state.growing && nq > state.prev_nq && (double)nq > na / 2000.0) state.forward = 0;
  state.prev_nq = nq;
  // The next top-down level needs this level's vertices as a queue, unless
  // the bottom-up body takes it.  A small level appended them to queue[qn];
  // a bulk one left them in vis[cur^1].
  if (!bulk) {
    state.qi = qn;
  } else if (state.forward &&
             !tail_pulls(1, state.growing, b.tail_pull, nq, g.n_active - state.visited)) {
    device_scan(FrontierBits{b.vis[cur ^ 1].p, nullptr}, FrontierEmit{b.vis[cur ^ 1].p, nullptr, b.queue[qi].p},
                (size_t)b.words, b.scan_tmp.p, s);
  }
}

// The frontier after a bottom-up level as a queue: vis[cur] & ~vis[cur ^ 1].
static void queue_from_bitmaps(BfsState& b, hipStream_t s, StepState& state) {
  const uint64_t *now = b.vis[state.cur].p, *before = b.vis[state.cur ^ 1].p;
  device_scan(FrontierBits{now, before}, FrontierEmit{now, before, b.queue[state.qi].p}, (size_t)b.words, b.scan_tmp.p,
              s);
  state.queued = 1;
  state.edges = 0;
}

// Bottom-up levels launched one by one, the next once the count of the last
// is known: on large graphs the round trip is small next to the level, and
// k_bu runs more waves than a step.  Returns before a top-down level that
// the top-down kernels take.
static void host_bottom_up(g5_ctx* ctx, BfsState& b, hipStream_t s, const StepArgs& a, StepState& state) {
  Graph& g = ctx->graph;
  unsigned long long* cnt = (unsigned long long*)b.counters.p;
  g5_bfs_stats& st = b.stats;
  while (state.nf && (!state.forward || tail_pulls(state.forward, state.growing, b.tail_pull, state.nf,
                                                   g.n_active - state.visited))) {
    const int lvl = state.lvl + 1;
    if (lvl > kStepMaxLevel) break;
    hipLaunchKernelGGL(k_bu, dim3(grid_of((b.words + a.span - 1) / a.span, kBlock / 64, 8192)), dim3(kBlock), 0, s, a,
                       state.cur, lvl, cnt, b.stamp.p);
    G5_HIP(hipGetLastError());
    ++b.pub_seq;
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, s, cnt, b.prefix.p, (int64_t)0, 0, b.pub.d, b.pub_seq,
                       b.stamp.p);
    G5_HIP(hipGetLastError());
    wait_published(b, s);
    const int64_t nq = (int64_t)b.h_counters[C_FOUND];
    st.direction[lvl] = state.forward;
    st.bu_kernel[lvl] = 1;
    st.nq[lvl] = nq;
    st.level_ms[lvl] = (double)b.h_counters[C_NUM] / (double)b.tick_khz;
    st.num_levels = lvl + 1;
    state.cur ^= 1;
    state.queued = 0;
    step_fold(g.n_active, state, nq);
  }
  state.stop = STEP_GO;
  if (state.nf && state.forward) queue_from_bitmaps(b, s, state);
}

// One workgroup takes the whole search of the smallest graphs.
static bool step_alone(const Graph& g, const BfsState& b) {
  return b.words <= kStepAloneWords && g.nnz <= kStepAloneEdges;
}
// Bitmap words per wave turn of a bottom-up level.  In a step, what gives
// every wave the same number of turns; for k_bu, 8, or 16 where a wave still
// has ten turns or more (S26 8/16: 674/685 us a search, S28: 2,521/2,469, before rows went to groups).
static int bottom_up_span(const Graph& g, const BfsState& b) {
  if (b.words == 0) return 1;  // a graph without rows has no turns to share out
  if (b.words > kStepMaxWords) return b.words >= (INT64_C(1) << 20) ? 16 : 8;
  const int64_t waves = (step_alone(g, b) ? 1 : kStepMaxGrid) * (kStepThreads / 64);
  const int64_t turns = (b.words + waves * kBuSpan - 1) / (waves * kBuSpan);
  return (int)((b.words + waves * turns - 1) / (waves * turns));
}
// Workgroups of a step: one for the smallest graphs; else enough waves for a
// turn of every wave in a bottom-up level, and at least kStepMinGrid for the
// top-down levels.
static unsigned step_grid(const Graph& g, const BfsState& b, int span) {
  if (step_alone(g, b)) return 1;
  return std::max(kStepMinGrid, grid_of((b.words + span - 1) / span, kStepThreads / 64, kStepMaxGrid));
}

// Steps until one stops; returns its state (see k_bfs_step).  k counts the
// search's steps; kStepAhead of them wait behind the running one.
static StepState run_steps(BfsState& b, hipStream_t s, unsigned grid, int lvl0, int& k) {
  const uint64_t seq = ++b.step_seq;
  const int k0 = k, ahead = grid == 1 ? 0 : kStepAhead;
  const PublishBlock& pub = b.step_pub;
  for (uint64_t spins = 1; !pub.ready(P_STOP, P_STOP + 1, seq); ++spins) {
    const int started = pub.ready(P_STEP, P_STEP + 1, seq) ? (int)pub.value(P_STEP) : k0;
    if (k - started < std::max(ahead, k == k0 ? 1 : 0) || k - k0 < ahead) {
      hipLaunchKernelGGL(k_bfs_step, dim3(grid), dim3(kStepThreads), 0, s, (unsigned long long*)b.step_ctl.p, k, seq);
      G5_HIP(hipGetLastError());
      ++k;
    } else if (spins % 4096 == 0) {
      const hipError_t e = hipStreamQuery(s);
      if (e == hipErrorNotReady) continue;
      G5_HIP(e);
      G5_CHECK(pub.ready(P_STEP, P_STEP + 1, seq), "g5_run_bfs: a step was not published");
    }
  }
  pub.wait(P_STOP, P_NUM, seq, s, "g5_run_bfs: the last step's state was not published");
  StepState r{};
  r.stop = (int32_t)pub.value(P_STOP);
  r.lvl = (int32_t)pub.value(P_LVL);
  const uint64_t bits = pub.value(P_BITS);
  r.forward = bits & 1;
  r.growing = (bits >> 1) & 1;
  r.cur = (bits >> 2) & 1;
  r.queued = (bits >> 3) & 1;
  r.qi = (int32_t)(bits >> 4);
  r.nf = (int64_t)pub.value(P_NF);
  r.prev_nq = (int64_t)pub.value(P_PREV);
  r.visited = (int64_t)pub.value(P_VISITED);
  r.edges = pub.value(P_EDGES);
  const double tick_ms = 1.0 / (double)b.tick_khz;
  g5_bfs_stats& st = b.stats;
  pub.wait(2 * (lvl0 + 1), 2 * (r.lvl + 1), seq, s, "g5_run_bfs: levels were not published");
  for (int l = lvl0 + 1; l <= r.lvl; ++l) {
    const uint64_t v = pub.value(2 * l);
    st.nq[l] = (int64_t)(v >> 2);
    st.direction[l] = v & 1;
    st.bu_kernel[l] = (v >> 1) & 1;
    st.level_ms[l] = (double)pub.value(2 * l + 1) * tick_ms;
    st.num_levels = l + 1;
  }
  st.device_ms = (double)pub.value(P_TICKS) * tick_ms;
  return r;
}

void bfs_run(g5_ctx* ctx, BfsState& b, hipStream_t s, int64_t root) {
  Graph& g = ctx->graph;
  G5_CHECK(b.prepared, "g5_run_bfs: call g5_prepare_bfs first");
  G5_CHECK(root >= 0 && root < g.n, "g5_run_bfs: root out of range");
  const int64_t rows = g.n_rows;
  unsigned long long* cnt = (unsigned long long*)b.counters.p;
  b.have_result = false;
  b.root_orig = root;
  g5_bfs_stats& st = b.stats;
  st = g5_bfs_stats{};

  if (b.hub_shift > 0 && b.hub_built_shift != b.hub_shift) bfs_tuning_buffers(ctx, b, s);

  StepArgs a{};
  a.offsets = g.offsets.p;
  a.cols = g.cols.p;
  a.first_nbr = g.first_nbr.p;
  for (int i = 0; i < 2; ++i) a.vis[i] = b.vis[i].p;
  for (int i = 0; i < 3; ++i) a.queue[i] = b.queue[i].p;
  a.level = b.level.p;
  a.parent = b.parent.p;
  a.pub = b.step_pub.d;
  a.words = b.words;
  a.n_active = g.n_active;
  a.small_edges = b.small_edges;
  a.tail_pull = b.tail_pull;
  a.host_bu = b.words > kStepMaxWords;
  a.span = bottom_up_span(g, b);
  a.share = b.words <= kStepShareWords;
  const unsigned grid = step_grid(g, b, a.span);
  // A root without edges (reachable only through a find_roots fallback) is
  // the whole tree: the reference's first top-down level finds nothing.
  const bool root_active = (g.has_edge_words[root >> 6] >> (root & 63)) & 1;
  hipLaunchKernelGGL(k_bfs_init, dim3(grid_of((rows + 15) / 16, kBlock, 2048)), dim3(kBlock), 0, s, g.old2new.p, root,
                     rows, b.words, b.level.p, b.parent.p, b.vis[0].p, b.queue[0].p,
                     (unsigned long long*)b.step_ctl.p, cnt, a, root_active ? 1 : 0);
  G5_HIP(hipGetLastError());

  StepState state{};
  state.visited = 1;
  int steps = 0;
  bool resume = false;  // the state has gone on in host code since the last step
  const auto bottom_up_next = [&] {
    return !state.forward ||
           tail_pulls(1, state.growing, b.tail_pull, state.nf, g.n_active - state.visited);
  };
  for (;;) {
    if (resume && state.nf && a.host_bu && bottom_up_next() && state.lvl < kStepMaxLevel) {
      host_bottom_up(ctx, b, s, a, state);
      continue;
    }
    if (resume && state.nf > kStepNf && !bottom_up_next() && state.lvl < kStepMaxLevel) {
      large_top_down(ctx, b, s, state);
      continue;
    }
    if (resume) {
      hipLaunchKernelGGL(k_step_resume, dim3(1), dim3(1), 0, s, (unsigned long long*)b.step_ctl.p, state, steps);
      G5_HIP(hipGetLastError());
    }
    state = run_steps(b, s, grid, state.lvl, steps);
    if (state.stop == STEP_DONE) break;
    G5_CHECK(state.stop != STEP_LIMIT, "g5_run_bfs: more than 254 levels (uint8 level array)");
    const int stop = state.stop;
    state.stop = STEP_GO;
    resume = true;
    if (!state.queued && stop != STEP_BOTTOM_UP) queue_from_bitmaps(b, s, state);
    if (stop == STEP_LARGE) large_top_down(ctx, b, s, state);
  }
  if (!root_active) {  // the level that finds nothing was not run
    st.num_levels = 2;
    st.direction[1] = 1;
  }
  st.reached = state.visited;
  b.have_result = true;
}

// Predecessors are 8 B an id, made faster than the link takes them, so large
// ones are bound by the link alone: 53 GB/s of a kernel's stores, 57 of the
// copy engine (S22/S24/S26: 664, 2,613 and 10,414 us stored, 646, 2,495 and
// 10,040 copied; S18, S20 and S21 51, 174 and 337 against 60, 180 and 337).
constexpr size_t kPredDirect = size_t(16) << 20;

void bfs_get_pred(g5_ctx* ctx, int64_t* host_pred) {
  Graph& g = ctx->graph;
  BfsState& b = ctx->bfs;
  G5_CHECK(b.have_result, "g5_get_pred: no BFS result (call g5_run_bfs first)");
  HostOut out(host_pred, (size_t)g.n, ctx->stage, b.pred_out, ctx->stream, kPredDirect);
  hipLaunchKernelGGL(k_make_pred, dim3(grid_of(g.n, kBlock, 65536)), dim3(kBlock), 0, ctx->stream,
                     g.old2new.p, g.new2old.p, b.level.p, b.parent.p, g.n, g.n_rows, b.root_orig, (int64_t*)out.p);
  G5_HIP(hipGetLastError());
  out.finish();
}

void bfs_get_levels(g5_ctx* ctx, uint8_t* host_levels) {
  Graph& g = ctx->graph;
  BfsState& b = ctx->bfs;
  G5_CHECK(b.have_result, "g5_get_levels: no BFS result (call g5_run_bfs first)");
  HostOut out(host_levels, (size_t)g.n, ctx->stage, b.level_out, ctx->stream);
  launch_make_levels(g.old2new.p, b.level.p, g.n, g.n_rows, b.root_orig, (uint8_t*)out.p, ctx->stream);
  out.finish();
}

int64_t bfs_teps_edges(g5_ctx* ctx) { return bfs_teps_edges(ctx, ctx->bfs, ctx->stream); }

int64_t bfs_teps_edges(g5_ctx* ctx, BfsState& b, hipStream_t s) {
  Graph& g = ctx->graph;
  G5_CHECK(b.have_result, "g5_teps_edges: no BFS result (call g5_run_bfs first)");
  const unsigned grid = grid_of((g.n_rows + 15) / 16, kTepsThreads, kTepsGrid);
  ++b.teps_seq;
  hipLaunchKernelGGL(k_teps, dim3(grid), dim3(kTepsThreads), 0, s, b.level.p, g.weight.p, g.n_rows, b.teps_pub.d,
                     b.teps_seq);
  G5_HIP(hipGetLastError());
  b.teps_pub.wait(0, (int)grid, b.teps_seq, s, "g5_teps_edges: a sum was not published");
  uint64_t sum = 0;
  for (unsigned i = 0; i < grid; ++i) sum += b.teps_pub.value(i);
  return (int64_t)(sum / 2);
}

}  // namespace g5
