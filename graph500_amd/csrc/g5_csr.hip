// g5_csr.hip -- CSR construction in HBM.
//
// Restates the semantics of GraphConstructor2DCSR::construct
// (mpi/graph_constructor.hpp:554-574) for one GPU:
//   searchMaxVertex      estimated SCALE = msb(OR of all ids) + 1      (:735-763)
//   scatterAndScanEdges  self loops dropped; degree counts duplicates  (:765-843)
//   calc_degree VR=2     vertices ordered by degree, descending        (:296-352)
//                        (ties by original id: stable sort, the
//                        reference's std::sort leaves them unspecified)
//   sortEdges            rows sorted by reordered target, duplicates removed (:1376-1442)
//   isolateFirstEdge     first (smallest new id) neighbour kept apart  (:845-879)
//   computeNumVertices   n_active = vertices with an edge              (:1444-1464)
//
// Device pipeline: OR-reduce -> directed entries grouped by vertex range ->
// degrees counted in LDS per range -> stable radix sort of (degree key, id) ->
// entries relabelled range by range, grouped by row ranges, then by estimated
// position, sorted and deduplicated in LDS (g5_entries.hpp).  The tuples
// themselves are never re-sorted.
#include "g5_answers.hpp"
#include "g5_ctx.hpp"
#include "g5_entries.hpp"
#include "g5_prims.hpp"

#include <algorithm>

namespace g5 {

__device__ __forceinline__ uint64_t tuple_v0(const g5_packed_edge& e) {
  return (uint64_t)e.v0_low | ((uint64_t)(e.high & 0xFFFF) << 32);
}
__device__ __forceinline__ uint64_t tuple_v1(const g5_packed_edge& e) {
  return (uint64_t)e.v1_low | ((uint64_t)(e.high >> 16) << 32);
}

// The OR of all ids, by workgroup: each publishes its own to the host, which
// combines them (atomics by every wave of a 65,536-workgroup grid spent 3 ms on
// one word, 12 ns each).
__global__ void __launch_bounds__(kBlock) k_or_ids(const g5_packed_edge* __restrict__ e, int64_t m,
                                                   Published* __restrict__ pub, uint64_t seq) {
  __shared__ uint64_t s_or[kBlock / 64];
  uint64_t acc = 0;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
#pragma unroll 4
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < m; i += stride) {
    const g5_packed_edge t = e[i];
    acc |= tuple_v0(t) | tuple_v1(t);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc |= __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) s_or[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / 64; ++w) acc |= s_or[w];
    publish(pub + blockIdx.x, acc, seq);
  }
}

// Zeroes two arrays (a fill call each is one launch or two).
__global__ void __launch_bounds__(kBlock) k_zero2(uint32_t* __restrict__ a, int64_t na, uint32_t* __restrict__ b,
                                                  int64_t nb) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x, stride = (int64_t)gridDim.x * kBlock;
  for (int64_t i = t; i < na; i += stride) a[i] = 0;
  for (int64_t i = t; i < nb; i += stride) b[i] = 0;
}

// The info words, and the columns in all rows, to the host.
__global__ void __launch_bounds__(64) k_publish_info(const unsigned long long* __restrict__ info,
                                                     const uint64_t* __restrict__ nnz, Published* __restrict__ pub,
                                                     uint64_t seq) {
  if (threadIdx.x < I_NUM) publish(pub + threadIdx.x, info[threadIdx.x], seq);
  if (threadIdx.x == I_NUM) publish(pub + I_NUM, *nnz, seq);
}

// Sort keys for the vertex order: smaller key first, stable by id.
__global__ void k_order_keys(const uint32_t* __restrict__ deg, int64_t n, uint32_t maxdeg, int mode,
                             uint32_t* __restrict__ keys, uint32_t* __restrict__ ids) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t d = deg[v];
    keys[v] = (mode == 2) ? (maxdeg - d) : (d == 0 ? 1u : 0u);
    ids[v] = (uint32_t)v;
  }
}

__global__ void k_iota(int64_t n, uint32_t* __restrict__ out) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x)
    out[v] = (uint32_t)v;
}

// Degree (duplicates counted) and tuple weight (degree + 2 * loops) per row.
__global__ void k_row_info(const uint32_t* __restrict__ new2old, const uint32_t* __restrict__ deg,
                           const uint32_t* __restrict__ loops, int64_t rows, uint32_t* __restrict__ row_deg,
                           uint32_t* __restrict__ w) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= rows;
       v += (int64_t)gridDim.x * blockDim.x) {
    if (v == rows) {
      row_deg[v] = 0;  // the prefix's last element, the total
      continue;
    }
    const uint32_t o = new2old[v], d = deg[o];
    row_deg[v] = d;
    w[v] = loops ? d + 2u * loops[o] : d;
  }
}

// --- sorted entries to rows, for graphs whose entries were sorted by radix ---
struct UniqueFlag {
  const uint64_t* keys;
  size_t nvalid;
  __device__ uint64_t operator()(size_t i) const {
    if (i >= nvalid) return 0;
    return (i == 0 || keys[i] != keys[i - 1]) ? 1 : 0;
  }
};

// Writes the column of every first occurrence and the row offsets of every
// row that starts at it (rows with no entries in between get the same start).
struct UniqueStore {
  const uint64_t* keys;
  size_t nvalid;
  int scale;
  uint32_t* cols;
  uint64_t* offsets;
  __device__ void operator()(size_t i, uint64_t pre) const {
    if (i >= nvalid) return;
    const uint64_t k = keys[i];
    if (i != 0 && k == keys[i - 1]) return;
    const uint64_t mask = (UINT64_C(1) << scale) - 1;
    cols[pre] = (uint32_t)(k & mask);
    const int64_t src = (int64_t)(k >> scale);
    const int64_t prev = (i == 0) ? -1 : (int64_t)(keys[i - 1] >> scale);
    for (int64_t r = prev + 1; r <= src; ++r) offsets[r] = pre;
  }
};

__global__ void k_offsets_tail(const uint64_t* __restrict__ keys, size_t nvalid, int scale,
                               int64_t rows, uint64_t nnz, uint64_t* __restrict__ offsets) {
  const int64_t last = nvalid ? (int64_t)(keys[nvalid - 1] >> scale) : -1;
  for (int64_t r = last + 1 + (int64_t)(blockIdx.x * blockDim.x + threadIdx.x); r <= rows;
       r += (int64_t)gridDim.x * blockDim.x)
    offsets[r] = nnz;
}

__global__ void k_first_nbr(const uint64_t* __restrict__ offsets, const uint32_t* __restrict__ cols,
                            int64_t rows, uint32_t* __restrict__ first) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < rows;
       v += (int64_t)gridDim.x * blockDim.x) {
    const uint64_t b = offsets[v], e = offsets[v + 1];
    first[v] = (e > b) ? cols[b] : 0xFFFFFFFFu;
  }
}

// has_edge bitmap by original id.
__global__ void __launch_bounds__(kBlock) k_has_edge_bits(const uint32_t* __restrict__ deg, int64_t n,
                                                          uint64_t* __restrict__ words,
                                                          const unsigned long long* __restrict__ info,
                                                          Published* __restrict__ pub, uint64_t seq) {
  // the host goes on with the info words while the bits are made
  if (blockIdx.x == 0 && threadIdx.x < I_NUM) publish(pub + threadIdx.x, info[threadIdx.x], seq);
  // a wave makes 16 words, stored together (they may go to the host's memory)
  const int lane = threadIdx.x & 63;
  const int64_t nw = (n + 63) / 64, waves = (int64_t)gridDim.x * (kBlock / 64);
  for (int64_t w0 = ((int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * 16; w0 < nw; w0 += waves * 16) {
    uint64_t mine = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int64_t v = (w0 + j) * 64 + lane;
      const uint64_t w = __ballot(v < n && deg[v] > 0);
      if (lane == j) mine = w;
    }
    if (lane < 16 && w0 + lane < nw) words[w0 + lane] = mine;
  }
}

static unsigned grid_for(int64_t n, int64_t per_block = kBlock) {
  int64_t b = (n + per_block - 1) / per_block;
  if (b > 65536) b = 65536;
  return (unsigned)(b > 0 ? b : 1);
}

// Ranges of vertex ids for the degree counts and the relabelling: up to
// kPartMax of at least 64 vertices; at least 256 where the ids allow, so that
// small graphs fill the chip, and beyond that as many as keep a range within
// one workgroup's LDS counters (kDegVerts).
static int range_bits(int scale) { return std::min(10, std::max(std::min(8, std::max(scale - 6, 0)), scale - 15)); }

// From here on both endpoints of an entry are relabelled in one pass by
// lookups of old2new wherever they fall; a larger table is looked up one side
// at a time with the entries grouped by that side, one more pass over the
// entries but no lookup past the L2 (4 MB per XCD).  Random lookups of a
// 128 MB table run at 55 G/s, 20 ms per 10^9, the pass takes 5 ms; in a table
// that fits the L2 they run at the pass's own rate.
constexpr int kRelabelBothScale = 20;

// Workgroups of a pass over the tuples that ends with atomics on shared words
// (12 ns each, one after another).
constexpr unsigned kTupleGrid = 1024;

// Positions per sub-bucket, as a shift: 2^11 as long as two partitions by
// about 512 reach it, 2^12 beyond (2^31 entries on).
static int sub_shift_for(uint64_t entries) { return entries >> 31 ? 12 : 11; }

// L1 buckets: stretches of 2^wshift positions, at most 512 of them, or
// kPartMax once a sub-bucket has 2^12 positions.
static int l1_shift(uint64_t entries, int sub) {
  const uint64_t most = sub == 11 ? 512 : kPartMax;
  int w = sub;
  while ((entries - 1) >> w >= most) ++w;
  return w;
}

// Persistent grid of the partition passes: one workgroup per CU.
static unsigned part_grid(int64_t tiles) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(tiles, 256)); }

template <class Src>
static void partition(const Src& src, unsigned long long* cursor, uint64_t* out, hipStream_t s) {
  const int64_t tiles = src.tiles();
  hipLaunchKernelGGL(k_partition<Src>, dim3(part_grid(tiles)), dim3(kPartThreads), 0, s, src, tiles, cursor, out);
  G5_HIP(hipGetLastError());
}

// What a construction publishes: the OR of the ids by workgroup, then the info
// words after the degrees and, with the columns' count, after the sort.
constexpr int kPubOr = (int)kTupleGrid;
// Up to this many ids the bitmap of used ones fits the pinned stage, and
// scratch is kept to the end instead of given back on the way (12 B an id).
constexpr int64_t kSmallIds = (int64_t)HostOut::kStageBytes * 8;

void build_graph(g5_ctx* ctx, int mode, bool release_edges) {
  G5_CHECK(mode >= 0 && mode <= 2, "g5_construct: reorder_mode must be 0, 1 or 2");
  G5_CHECK(ctx->num_edges > 0, "g5_construct: the edge list is empty");
  hipStream_t s = ctx->stream;
  Graph& g = ctx->graph;
  g.clear();
  ctx->acc.alloc(4);
  const int64_t m = ctx->num_edges;
  const g5_packed_edge* e = ctx->edges.p;

  // What the host needs on the way is published to it (the OR of the ids by
  // workgroup, the info words twice); a copy and a wait each took 25 us more.
  ctx->build_pub.alloc_once(kPubOr + 2 * (I_NUM + 1));
  PublishBlock& pub = ctx->build_pub;
  const uint64_t seq = ++ctx->build_seq;
  hipEvent_t t0, t1;
  G5_HIP(hipEventCreate(&t0));
  G5_HIP(hipEventCreate(&t1));
  G5_HIP(hipEventRecord(t0, s));

  // 1. estimated SCALE
  const unsigned or_grid = std::min(grid_for(m, kBlock * 8), kTupleGrid);
  hipLaunchKernelGGL(k_or_ids, dim3(or_grid), dim3(kBlock), 0, s, e, m, pub.d, seq);
  G5_HIP(hipGetLastError());
  pub.wait(0, (int)or_grid, seq, s, "g5_construct: the ids' bits were not published");
  uint64_t orv = 0;
  for (unsigned i = 0; i < or_grid; ++i) orv |= pub.value((int)i);
  int scale = 0;
  while (scale < 64 && (orv >> scale)) ++scale;
  G5_CHECK(scale >= 1, "g5_construct: all vertex ids are zero");
  if (scale > 32) throw Error{"g5_construct: vertex ids need " + std::to_string(scale) +
                              " bits; this build supports up to 2^32 vertices"};
  const int64_t n = (int64_t)1 << scale;
  g.scale = scale;
  g.n = n;
  g.num_tuples = m;
  g.reorder_mode = mode;

  // 2. directed entries grouped by ranges of 2^shift ids, and the degrees
  // (duplicates counted, loops apart)
  const int shift = scale - range_bits(scale), nb = 1 << range_bits(scale);
  const int sub_shift = std::min(shift, 15);
  static_assert(kDegVerts == 1 << 15, "one workgroup counts 2^15 vertices");
  DevBuf<uint32_t> deg, loops;
  deg.alloc(n);
  loops.alloc(n);
  // counts | cursors of the two range partitions | of the row partition, then bucket bounds and the info words
  DevBuf<unsigned long long> ctl;
  const size_t pad = (size_t)kPartMax * kCursorPad;
  ctl.alloc(4 * pad + 2 * (kPartMax + 1) + I_NUM);
  unsigned long long *counts = ctl.p, *cur0 = ctl.p + pad, *cur1 = cur0 + pad, *cur2 = cur1 + pad;
  uint64_t* range_off = (uint64_t*)(cur2 + pad);
  uint64_t* l1_base = range_off + kPartMax + 1;
  unsigned long long* info = cur2 + pad + 2 * (kPartMax + 1);
  hipLaunchKernelGGL(k_zero2, dim3(grid_for(std::max<int64_t>(n, (int64_t)ctl.n * 2), kBlock * 4)), dim3(kBlock), 0, s,
                     (uint32_t*)ctl.p, (int64_t)ctl.n * 2, loops.p, n);
  hipLaunchKernelGGL(k_part_count, dim3(std::min(grid_for(m, kBlock * 8), kTupleGrid)), dim3(kBlock), 0, s, e, m, shift, nb,
                     counts, info);
  hipLaunchKernelGGL(k_part_offsets, dim3(1), dim3(kPartMax), 0, s, counts, nb, range_off, cur0, cur1);
  const size_t nkeys = 2 * (size_t)m;
  DevBuf<uint64_t> xa, xb;
  xa.alloc(nkeys);
  partition(SrcTuples{e, m, loops.p, shift}, cur0, xa.p, s);
  hipLaunchKernelGGL(k_bucket_degrees, dim3((unsigned)nb << (shift - sub_shift)), dim3(1024), 0, s, xa.p, range_off,
                     shift, sub_shift, n, deg.p, info);
  // has_edge bitmap by original id, kept on the host for root selection; small
  // ones are written to pinned host memory by the kernel
  DevBuf<uint64_t> words;
  const int64_t nw = (n + 63) / 64;
  const bool small = n <= kSmallIds;
  uint64_t* h_words = nullptr;
  if (small) {
    h_words = (uint64_t*)ctx->stage.get(HostOut::kStageBytes);
  } else {
    words.alloc(nw);
  }
  hipLaunchKernelGGL(k_has_edge_bits, dim3(grid_for(n, kBlock * 16)), dim3(kBlock), 0, s, deg.p, n, small ? h_words : words.p, info,
                     pub.d + kPubOr, seq);
  G5_HIP(hipGetLastError());
  uint64_t h_info[I_NUM];
  const auto read_info = [&](int at, int count) {
    pub.wait(at, at + count, seq, s, "g5_construct: counts were not published");
    for (int i = 0; i < I_NUM; ++i) h_info[i] = pub.value(at + i);
  };
  read_info(kPubOr, I_NUM);
  g.max_degree = (int64_t)h_info[I_MAXDEG];
  g.self_loops = (int64_t)h_info[I_LOOPS];
  g.n_active = (int64_t)h_info[I_ACTIVE];
  g.directed_before = 2 * (m - g.self_loops);
  g.n_rows = (mode == 0) ? n : g.n_active;
  if (release_edges && !small) {
    ctx->edges.release();
    ctx->num_edges = 0;
  }
  g.has_edge_words.resize(nw);
  if (!small) {
    G5_HIP(hipMemcpyAsync(g.has_edge_words.data(), words.p, nw * 8, hipMemcpyDeviceToHost, s));
    G5_HIP(hipStreamSynchronize(s));
    words.drop();
  }

  // 3. vertex order
  g.new2old.alloc(n);
  g.old2new.alloc(n);
  RadixScratch rs;
  DevBuf<uint32_t> k0, k1, v1;
  if (mode == 0) {
    hipLaunchKernelGGL(k_iota, dim3(grid_for(n)), dim3(kBlock), 0, s, n, g.new2old.p);
    G5_HIP(hipGetLastError());
  } else {
    k0.alloc(n);
    k1.alloc(n);
    v1.alloc(n);
    hipLaunchKernelGGL(k_order_keys, dim3(grid_for(n)), dim3(kBlock), 0, s, deg.p, n,
                       (uint32_t)g.max_degree, mode, k0.p, g.new2old.p);
    G5_HIP(hipGetLastError());
    int bits = 0;
    const uint64_t kmax = (mode == 2) ? (uint64_t)g.max_degree : 1;
    while (bits < 32 && (kmax >> bits)) ++bits;
    uint32_t *kp = k0.p, *ka = k1.p, *vp = g.new2old.p, *va = v1.p;
    radix_sort_pairs_u32(&kp, &ka, &vp, &va, (size_t)n, 0, bits, rs, s);
    if (vp != g.new2old.p) g.new2old.swap(v1);
    if (!small) {  // the memory is needed below
      G5_HIP(hipStreamSynchronize(s));
      k0.drop();
      k1.drop();
      v1.drop();
    }
  }
  const int64_t rows = g.n_rows;
  g.weight.alloc(rows);
  g.offsets.alloc(rows + 1);
  DevBuf<uint32_t> row_cnt;  // degrees with duplicates, then unique entries per row
  DevBuf<uint64_t> P, tmp;   // degree prefix: P[r] = entries of the rows before r
  row_cnt.alloc(rows + 1);
  P.alloc(rows + 1);
  tmp.alloc(scan_tmp_elems(rows + 1));
  hipLaunchKernelGGL(k_row_info, dim3(grid_for(rows + 1)), dim3(kBlock), 0, s, g.new2old.p, deg.p,
                     g.self_loops ? loops.p : nullptr, rows, row_cnt.p, g.weight.p);
  G5_HIP(hipGetLastError());
  device_scan(LoadU32{row_cnt.p}, StoreU64{P.p}, (size_t)rows + 1, tmp.p, s);
  DevBuf<uint64_t> row_word;
  row_word.alloc(n);
  hipLaunchKernelGGL(k_row_words, dim3(grid_for(n)), dim3(kBlock), 0, s, g.new2old.p, n, P.p, rows, g.old2new.p,
                     row_word.p);
  G5_HIP(hipGetLastError());

  // 4. entries to sorted, deduplicated rows
  const uint64_t E = (uint64_t)g.directed_before;
  // Where the device is short, a request is tried again once the scratch that
  // no later pass reads has gone back; else that stays to the end, from where
  // the next construction takes it (given back earlier, it left the pool in an
  // order in which a repeated SCALE 26 build waits for the driver to clear
  // memory: 100 ms, then 0.4-1.5 s).
  std::vector<DevBuf<uint32_t>*> idle32{&deg, &loops};
  std::vector<DevBuf<uint64_t>*> idle64;
  const auto alloc = [&](auto& buf, size_t count) {
    try {
      buf.alloc(count);
    } catch (const Error& err) {
      if (err.code != G5_ERR_MEM) throw;
      G5_HIP(hipStreamSynchronize(s));
      for (DevBuf<uint32_t>* b : idle32) b->drop();
      for (DevBuf<uint64_t>* b : idle64) b->drop();
      buf.alloc(count);
    }
  };
  alloc(xb, nkeys);
  uint64_t nnz = 0;
  DevBuf<uint64_t> sub64;  // first position | first entry | first unique column
  DevBuf<uint32_t> sub32;  // entries | first row | unique columns | L1 first sub-buckets | column shares
  DevBuf<uint64_t> stmp;
  if (E == 0) {
    g.cols.alloc(0);
    G5_HIP(hipMemsetAsync(g.offsets.p, 0, (rows + 1) * 8, s));
  } else {
    const int sub = sub_shift_for(E), wshift = l1_shift(E, sub);
    const int nb1 = (int)(((E - 1) >> wshift) + 1);
    const size_t max_subs = (size_t)(E >> sub) + nb1 + 1;
    alloc(sub64, 3 * (max_subs + 1));
    alloc(sub32, 3 * max_subs + kPartMax + 1 + kFracMax);
    uint64_t *sub_pos = sub64.p, *sub_off = sub_pos + max_subs + 1, *out_off = sub_off + max_subs + 1;
    uint32_t *sub_cnt = sub32.p, *sub_row = sub_cnt + max_subs, *sub_unique = sub_row + max_subs;
    uint32_t *l1_sub0 = sub_unique + max_subs, *frac = l1_sub0 + kPartMax + 1;
    int flat = -1;  // degree order: share samples by octave
    if (mode != 2) {
      flat = 0;
      while (((rows - 1) >> flat) >= 4096) ++flat;
    }
    int sh = 0;
    const int frac_count = (int)FracMap::index((uint32_t)(rows - 1), flat, sh) + 2;
    G5_CHECK(frac_count <= kFracMax && nb1 <= kPartMax, "g5_construct: share table or bucket count too small");
    hipLaunchKernelGGL(k_frac_table, dim3(grid_for(frac_count)), dim3(kBlock), 0, s, P.p, rows, flat, frac_count, frac);
    hipLaunchKernelGGL(k_l1_setup, dim3(1), dim3(kPartMax), 0, s, P.p, rows, wshift, sub, nb1, l1_base, l1_sub0, cur2,
                       sub_pos, info);
    hipLaunchKernelGGL(k_sub_rows, dim3(std::min(grid_for(rows), 4096u)), dim3(kBlock), 0, s, P.p, rows, wshift, sub,
                       l1_base, l1_sub0, info, sub_row);
    G5_HIP(hipGetLastError());
    uint64_t *grouped, *refined;  // entries by L1 bucket (kept until the sort is known to have fit), by sub-bucket
    if (scale <= kRelabelBothScale) {
      grouped = xb.p;
      refined = xa.p;
      partition(SrcPosition<true>{xa.p, (int64_t)E, g.old2new.p, row_word.p, l1_base, nb1, wshift, frac, frac_count,
                                  flat}, cur2, grouped, s);
    } else {
      grouped = xa.p;
      refined = xb.p;
      partition(SrcRelabel{xa.p, (int64_t)E, g.old2new.p, shift}, cur1, xb.p, s);
      partition(SrcPosition<false>{xb.p, (int64_t)E, g.old2new.p, row_word.p, l1_base, nb1, wshift, frac, frac_count,
                                   flat}, cur2, grouped, s);
    }
    hipLaunchKernelGGL(k_refine, dim3((unsigned)nb1), dim3(1024), 0, s, grouped, refined, sub, l1_base, l1_sub0,
                       sub_pos, sub_off, sub_cnt, info);
    hipLaunchKernelGGL(k_zero2, dim3(grid_for(rows + 1, kBlock * 4)), dim3(kBlock), 0, s, row_cnt.p, rows + 1,
                       (uint32_t*)nullptr, (int64_t)0);
    if (sub == 11)
      hipLaunchKernelGGL(k_sort_sub<11>, dim3((unsigned)max_subs), dim3(SubSort<11>::kThreads), 0, s, refined, sub_off,
                         sub_cnt, sub_pos, sub_row, P.p, rows, row_cnt.p, sub_unique, info);
    else
      hipLaunchKernelGGL(k_sort_sub<12>, dim3((unsigned)max_subs), dim3(SubSort<12>::kThreads), 0, s, refined, sub_off,
                         sub_cnt, sub_pos, sub_row, P.p, rows, row_cnt.p, sub_unique, info);
    G5_HIP(hipGetLastError());
    alloc(stmp, scan_tmp_elems(max_subs));
    device_scan(LoadU32{row_cnt.p}, StoreU64{g.offsets.p}, (size_t)rows + 1, tmp.p, s);
    device_scan(LoadU32{sub_unique}, StoreU64{out_off}, max_subs, stmp.p, s);
    hipLaunchKernelGGL(k_publish_info, dim3(1), dim3(64), 0, s, info, g.offsets.p + rows, pub.d + kPubOr + I_NUM + 1,
                       seq);
    G5_HIP(hipGetLastError());
    read_info(kPubOr + I_NUM + 1, I_NUM + 1);
    nnz = pub.value(kPubOr + 2 * I_NUM + 1);
    if (!h_info[I_WIDE] && !h_info[I_OVERFLOW]) {
      idle64 = {refined == xa.p ? &xb : &xa, &row_word, &P, &tmp};
      alloc(g.cols, nnz);
      hipLaunchKernelGGL(k_compact, dim3((unsigned)max_subs), dim3(kBlock), 0, s, refined, sub_off, sub_unique, out_off,
                         info, g.cols.p);
      G5_HIP(hipGetLastError());
    } else {
      // Rows whose columns crowd into few positions (very long rows, many
      // copies of one tuple): the entries, still whole in `grouped`, are
      // sorted by radix instead.
      hipLaunchKernelGGL(k_entry_keys, dim3(grid_for((int64_t)E)), dim3(kBlock), 0, s, grouped, E, P.p, rows, l1_base,
                         nb1, refined);
      uint64_t *kp = refined, *ka = grouped;
      radix_sort_u64(&kp, &ka, E, 0, scale, rs, s);
      radix_sort_u64(&kp, &ka, E, 32, 32 + scale, rs, s);
      const UniqueFlag flag{kp, (size_t)E};
      nnz = device_reduce_sum(flag, E, ctx->acc.p, s);
      idle64 = {kp == xa.p ? &xb : &xa, &row_word, &P, &tmp};
      alloc(g.cols, nnz);
      alloc(stmp, scan_tmp_elems(E));
      device_scan(flag, UniqueStore{kp, (size_t)E, 32, g.cols.p, g.offsets.p}, E, stmp.p, s);
      hipLaunchKernelGGL(k_offsets_tail, dim3(grid_for(rows)), dim3(kBlock), 0, s, kp, (size_t)E, 32, rows, nnz,
                         g.offsets.p);
      G5_HIP(hipGetLastError());
    }
  }
  g.nnz = (int64_t)nnz;

  idle32 = {&deg, &loops, &row_cnt, &sub32};
  idle64 = {&xa, &xb, &row_word, &P, &tmp, &sub64, &stmp};
  alloc(g.first_nbr, rows);
  hipLaunchKernelGGL(k_first_nbr, dim3(grid_for(rows)), dim3(kBlock), 0, s, g.offsets.p, g.cols.p,
                     rows, g.first_nbr.p);
  G5_HIP(hipGetLastError());
  G5_HIP(hipEventRecord(t1, s));
  G5_HIP(hipEventSynchronize(t1));
  float ms = 0;
  G5_HIP(hipEventElapsedTime(&ms, t0, t1));
  g.construct_ms = ms;
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  // all work is done: the scratch goes back without a wait each
  if (small) std::copy(h_words, h_words + nw, g.has_edge_words.begin());
  g.max_used_vertex = 0;
  for (int64_t w = nw - 1; w >= 0; --w)
    if (g.has_edge_words[w]) {
      g.max_used_vertex = w * 64 + 63 - __builtin_clzll(g.has_edge_words[w]);
      break;
    }
  if (release_edges && small) {
    ctx->edges.drop();
    ctx->num_edges = 0;
  }
  for (DevBuf<uint32_t>* b : {&deg, &loops, &k0, &k1, &v1, &row_cnt, &sub32}) b->drop();
  for (DevBuf<uint64_t>* b : {&xa, &xb, &P, &tmp, &row_word, &sub64, &stmp}) b->drop();
  ctl.drop();
  g.built = true;
}

}  // namespace g5
