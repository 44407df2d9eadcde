// moe_align / permute: per-expert counts, offsets and a stable expert-major
// permutation of the routed (token, slot) pairs, in one workgroup (or, for large batches
// with a workspace, in two launches over many workgroups).
//
// Replaces, at ep=1:
//   _MoeBlock._all_expert_count_compute (easyinfra/generation/blocks/moe/base.py:343-364)
//     counts = zeros(E).scatter_add_(0, ids, 1), restricted to the local window (base.py:187)
//   MoeAll2AllBlock.all2all_chunk_routing_compute (moe_all2all.py:346-348)
//     idx = ids.view(-1).sort().indices; token = idx // k; slot = idx % k
// and the M-block schedule of TritonExperts.forward_ep (fused_moe.py:413-439): the
// GEMMs derive their tiles from ``offsets`` on the device, so no host sync is needed.
//
// Order is pinned stable: (expert, flat index t*k+slot).  Integer-only and bit-exact.
//
// Algorithm (16 waves, LDS counting sort): wave w owns a contiguous slice of the
// flat ids.  Pass 1 builds a per-wave histogram with match masks (8-10 ballots per
// 64 ids, no atomics).  A prefix over waves and experts turns it into per-(wave,
// expert) write cursors.  Pass 2 re-reads the slice; each id's slot is its cursor
// plus its rank among equal ids below it in the wave, so the result is stable.
// Both passes fetch kAlignBatch rows of 64 ids per lane before using any of them: one
// workgroup does all the work, so a dependent load per 64 ids would put a memory
// latency on every step (tens of microseconds at 16-25k routed pairs).
#include "kernels.h"
#include "routing.h"

namespace eimoe {

__global__ __launch_bounds__(kAlignThreads) void align_kernel(const int32_t* __restrict__ ids, int N, int k,
                                                              int e_lo, int n_loc, int32_t* __restrict__ counts,
                                                              int32_t* __restrict__ offsets,
                                                              int32_t* __restrict__ sorted_flat,
                                                              int32_t* __restrict__ sorted_tok,
                                                              int32_t* __restrict__ pos) {
  extern __shared__ int lds[];
  align_rows<false>(ids, N, k, e_lo, n_loc, counts, offsets, sorted_flat, sorted_tok, pos, lds);
}

// ---------------------------------------------------------------------------- many workgroups
// Large batches: the same counting sort on B workgroups of kAlignMbWaves waves, workgroup
// b owning the contiguous chunk [b*chunk, (b+1)*chunk) of the flat ids (each wave a
// quarter of it).  align_hist_kernel writes every chunk's per-expert counts to
// hist[B][n_loc]; align_place_kernel has each workgroup sum that matrix (the totals, and
// per expert the counts of the chunks before its own: its chunk's base), recount its
// chunk per wave and place its ids.  Chunks precede each other in flat order, so the
// order is the same stable (expert, flat index) order; workgroup 0 writes counts and
// offsets.
constexpr int kAlignMbWaves = 4;
constexpr int kAlignMbThreads = 64 * kAlignMbWaves;

__global__ __launch_bounds__(kAlignMbThreads) void align_hist_kernel(const int32_t* __restrict__ ids, int N, int e_lo,
                                                                     int n_loc, int chunk,
                                                                     int32_t* __restrict__ hist_g) {
  extern __shared__ int lds[];   // [kAlignMbWaves][n_loc]
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int nbits = n_loc > 1 ? 32 - __clz(n_loc - 1) : 0;
  for (int i = tid; i < kAlignMbWaves * n_loc; i += kAlignMbThreads) lds[i] = 0;
  __syncthreads();
  const int sub = chunk / kAlignMbWaves;
  const long long beg = static_cast<long long>(blockIdx.x) * chunk + static_cast<long long>(w) * sub;
  if (beg < N) count_slice<false>(ids, static_cast<int>(beg), static_cast<int>(min<long long>(N, beg + sub)), e_lo, n_loc,
                                  nbits, lds + w * n_loc);
  __syncthreads();
  for (int e = tid; e < n_loc; e += kAlignMbThreads) {
    int c = 0;
#pragma unroll
    for (int ww = 0; ww < kAlignMbWaves; ++ww) c += lds[ww * n_loc + e];
    hist_g[static_cast<long long>(blockIdx.x) * n_loc + e] = c;
  }
}

__global__ __launch_bounds__(kAlignMbThreads) void align_place_kernel(
    const int32_t* __restrict__ ids, int N, int k, int e_lo, int n_loc, int chunk, const int32_t* __restrict__ hist_g,
    int32_t* __restrict__ counts, int32_t* __restrict__ offsets, int32_t* __restrict__ sorted_flat,
    int32_t* __restrict__ sorted_tok, int32_t* __restrict__ pos) {
  extern __shared__ int lds[];
  int* hist = lds;                                // [kAlignMbWaves][n_loc]
  int* tot = hist + kAlignMbWaves * n_loc;        // [n_loc]
  int* base = tot + n_loc;                        // [n_loc]
  int* offs = base + n_loc;                       // [n_loc + 1]
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int nbits = n_loc > 1 ? 32 - __clz(n_loc - 1) : 0;
  for (int i = tid; i < kAlignMbWaves * n_loc; i += kAlignMbThreads) hist[i] = 0;
  for (int e = tid; e < n_loc; e += kAlignMbThreads) tot[e] = base[e] = 0;
  __syncthreads();
  // Column sums of the chunk-count matrix (at most kAlignMbMaxCells cells, coalesced): totals, and the
  // chunks before this one.  A thread sums one expert's cells of every groups-th chunk in registers and
  // adds them to LDS once (integers, so the order does not matter).  The first few cells per thread are
  // loaded before the recount below, so their latency overlaps it.
  const int rows = static_cast<int>(gridDim.x);
  const int own = static_cast<int>(blockIdx.x);
  const int cols = min(n_loc, kAlignMbThreads);
  const int groups = kAlignMbThreads / cols;
  const int col = tid % cols;
  const int r0 = tid / cols < groups ? tid / cols : rows;
  constexpr int kEarly = 8;
  int early[kEarly];
#pragma unroll
  for (int j = 0; j < kEarly; ++j) {
    const int r = r0 + j * groups;
    early[j] = r < rows ? hist_g[r * n_loc + col] : 0;
  }
  const int sub = chunk / kAlignMbWaves;
  const long long beg = static_cast<long long>(blockIdx.x) * chunk + static_cast<long long>(w) * sub;
  const int b0 = static_cast<int>(min<long long>(beg, N));
  const int b1 = static_cast<int>(min<long long>(beg + sub, N));
  count_slice<false>(ids, b0, b1, e_lo, n_loc, nbits, hist + w * n_loc);
  for (int e = col; e < n_loc; e += cols) {
    int t = 0, before = 0;
    int r = r0;
    if (e == col) {
#pragma unroll
      for (int j = 0; j < kEarly; ++j) {
        t += early[j];
        before += r0 + j * groups < own ? early[j] : 0;
      }
      r += kEarly * groups;
    }
#pragma unroll 8
    for (; r < rows; r += groups) {
      const int c = hist_g[r * n_loc + e];
      t += c;
      before += r < own ? c : 0;
    }
    if (t != 0) atomicAdd(&tot[e], t);
    if (before != 0) atomicAdd(&base[e], before);
  }
  __syncthreads();
  scan_experts(tot, n_loc, offs);
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int e = tid; e < n_loc; e += kAlignMbThreads) counts[e] = tot[e];
    for (int i = tid; i <= n_loc; i += kAlignMbThreads) offsets[i] = offs[i];
  }
  // per-(wave, expert) cursors: expert start + chunks before this one + waves before this one
  for (int e = tid; e < n_loc; e += kAlignMbThreads) {
    int c = offs[e] + base[e];
#pragma unroll
    for (int ww = 0; ww < kAlignMbWaves; ++ww) {
      const int n = hist[ww * n_loc + e];
      hist[ww * n_loc + e] = c;
      c += n;
    }
  }
  __syncthreads();
  place_slice<false>(ids, b0, b1, k, e_lo, n_loc, nbits, hist + w * n_loc, sorted_flat, sorted_tok, pos);
}

size_t align_lds_bytes(int n_loc) { return static_cast<size_t>(align_lds_ints(n_loc)) * sizeof(int); }

hipError_t launch_align_place(const int32_t* ids, int T, int k, int e_lo, int n_loc, int blocks, int chunk,
                              const int32_t* hist, int32_t* counts, int32_t* offsets, int32_t* sorted_flat,
                              int32_t* sorted_tok, int32_t* pos, hipStream_t s) {
  if (blocks < 1 || chunk % kAlignMbWaves != 0 || static_cast<long long>(blocks) * n_loc > kAlignMbMaxCells)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(align_place_kernel, dim3(blocks), dim3(kAlignMbThreads),
                     static_cast<size_t>(kAlignMbWaves + 3) * n_loc * sizeof(int) + sizeof(int), s, ids, T * k, k, e_lo,
                     n_loc, chunk, hist, counts, offsets, sorted_flat, sorted_tok, pos);
  return hipGetLastError();
}

AlignPlan align_plan(int N, int n_loc) {
  AlignPlan pl{};
  if (N < kAlignMbMinIds) return pl;
  const int per = kAlignMbIdsPerBlock;
  int blocks = (N + per - 1) / per;
  if (blocks > kAlignMbMaxBlocks) blocks = kAlignMbMaxBlocks;
  if (blocks > kAlignMbMaxCells / n_loc) blocks = kAlignMbMaxCells / n_loc;   // each workgroup reads the matrix
  if (blocks < 1) blocks = 1;
  int chunk = (N + blocks - 1) / blocks;
  chunk = (chunk + 64 * kAlignMbWaves - 1) / (64 * kAlignMbWaves) * (64 * kAlignMbWaves);
  pl.blocks = (N + chunk - 1) / chunk;
  pl.chunk = chunk;
  pl.hist_ints = static_cast<size_t>(pl.blocks) * n_loc;
  return pl;
}

hipError_t launch_align(const int32_t* ids, int T, int k, int e_lo, int n_loc, int32_t* counts, int32_t* offsets,
                        int32_t* sorted_flat, int32_t* sorted_tok, int32_t* pos, int32_t* hist, hipStream_t s) {
  const int N = T * k;
  const AlignPlan pl = align_plan(N, n_loc);
  if (hist != nullptr && pl.blocks > 0) {
    hipLaunchKernelGGL(align_hist_kernel, dim3(pl.blocks), dim3(kAlignMbThreads),
                       static_cast<size_t>(kAlignMbWaves) * n_loc * sizeof(int), s, ids, N, e_lo, n_loc, pl.chunk, hist);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_align_place(ids, T, k, e_lo, n_loc, pl.blocks, pl.chunk, hist, counts, offsets, sorted_flat,
                              sorted_tok, pos, s);
  }
  const size_t lds = align_lds_bytes(n_loc);
  hipLaunchKernelGGL(align_kernel, dim3(1), dim3(kAlignThreads), lds, s, ids, N, k, e_lo, n_loc, counts,
                     offsets, sorted_flat, sorted_tok, pos);
  return hipGetLastError();
}

// Segments from a counts vector (the forward_ep entry: rows already grouped by
// (src_rank, local_expert), fused_moe.py:395-439).  offsets = exclusive cumsum.
// ROWS: of segments over max_rows rows, where a negative count is an empty segment and the bounds end at
// max_rows (sums saturate there: with at most 2^24 rows, 2 GiB of 64 columns, nothing leaves 32 bits); the rows
// past the last segment get tail_words words of zeros each in tail.
template <bool ROWS>
__global__ __launch_bounds__(64) void counts_to_offsets_kernel(const int32_t* __restrict__ counts, int S,
                                                               int32_t* __restrict__ offsets, int max_rows,
                                                               uint32_t* __restrict__ tail, int tail_words) {
  const int lane = threadIdx.x;
  const int per = (S + 63) / 64;
  const int b0 = lane * per;
  auto count = [&](int s) { return ROWS ? min(max(counts[s], 0), max_rows) : counts[s]; };
  auto bound = [&](int v) { return ROWS ? min(v, max_rows) : v; };
  int s = 0;
  for (int j = 0; j < per; ++j)
    if (b0 + j < S) s = bound(s + count(b0 + j));
  const int incl = wave_incl_scan(s);
  int run = incl - s;
  for (int j = 0; j < per; ++j) {
    if (b0 + j < S) {
      offsets[b0 + j] = bound(run);
      run = bound(run) + count(b0 + j);
    }
  }
  const int end = bound(__shfl(incl, 63, 64));
  if (lane == 63) offsets[S] = end;
  if constexpr (ROWS)
    for (int r = end; r < max_rows; ++r)
      for (int i = lane; i < tail_words; i += 64) tail[static_cast<long long>(r) * tail_words + i] = 0u;
}

hipError_t launch_counts_to_offsets(const int32_t* counts, int S, int32_t* offsets, hipStream_t s) {
  hipLaunchKernelGGL(counts_to_offsets_kernel<false>, dim3(1), dim3(64), 0, s, counts, S, offsets, 0, nullptr, 0);
  return hipGetLastError();
}

hipError_t launch_segment_bounds(const int32_t* counts, int S, int max_rows, int32_t* offsets, void* tail,
                                 int tail_bytes, hipStream_t s) {
  if (max_rows > (1 << 24)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(counts_to_offsets_kernel<true>, dim3(1), dim3(64), 0, s, counts, S, offsets, max_rows,
                     static_cast<uint32_t*>(tail), tail_bytes / 4);
  return hipGetLastError();
}

// Segments (source rank, expert) regrouped by expert.  Rows arrive grouped by source rank, then
// expert: segment s = rank * n_exp + e holds counts[s] rows.  A grouped GEMM over those segments
// reads each expert's weights once per rank and pads one tile per (rank, expert); merged, each
// expert is one segment.  offsets[n_exp + 1]: the experts' bounds in merged order; rows[m]: the
// original row of merged row m; pos[r]: the merged row of original row r, -1 for rows past the last
// segment, of which tail (null: left as it is) gets tail_words words of zeros each.  One launch (it stands
// in for counts_to_offsets, ~4.5 us either way).
// A negative count stands for an empty segment and the bounds end at max_rows, so that segments never
// overlap: every entry of pos is written, and every merged row below offsets[n_exp] names a row below
// max_rows, whatever the counts say.
// Workgroup s copies segment s's run; each recomputes the prefix sums of the (at most 1024) counts.
__global__ __launch_bounds__(256) void merge_segments_kernel(const int32_t* __restrict__ counts, int S, int n_exp,
                                                             int max_rows, int32_t* __restrict__ offsets,
                                                             int32_t* __restrict__ rows, int32_t* __restrict__ pos,
                                                             uint32_t* __restrict__ tail, int tail_words) {
  constexpr int kPer = 4;   // segments per thread: 256 * 4 = kMaxSeg
  static_assert(256 * kPer >= kMaxSeg, "one pass over the segments");
  __shared__ int s_wave[4];
  __shared__ int s_bound[256 * kPer + 1];
  __shared__ int s_red[4];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = tid >> 6;
  const int seg = blockIdx.x;
  int c[kPer];
  int sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int s = tid * kPer + j;
    c[j] = s < S ? min(max(counts[s], 0), max_rows) : 0;
    sum = min(sum + c[j], max_rows);
  }
  // Sums past max_rows stay there: with at most 2^24 rows (2 GiB of 64 columns) nothing leaves 32 bits.
  const int incl = wave_incl_scan(sum);
  if (lane == 63) s_wave[wv] = min(incl, max_rows);
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wv; ++w) run += s_wave[w];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    s_bound[tid * kPer + j] = min(run, max_rows);
    run += c[j];
  }
  if (tid == 255) s_bound[256 * kPer] = min(run, max_rows);
  __syncthreads();
  const int end = s_bound[S];
  if (tail)
    for (int r = end + seg; r < max_rows; r += gridDim.x)
      for (int i = tid; i < tail_words; i += 256) tail[static_cast<long long>(r) * tail_words + i] = 0u;
  // of this thread's segments, the rows of those before `seg` in merged order (a lower expert, or the same
  // expert of a lower rank)
  const int e = seg % n_exp;
  int before = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int s = tid * kPer + j;
    if (s >= S) continue;
    const int es = s % n_exp;
    if (es < e || (es == e && s < seg)) before += s_bound[s + 1] - s_bound[s];
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) before += __shfl_xor(before, m, 64);
  if (lane == 0) s_red[wv] = before;
  __syncthreads();
  const int dst = s_red[0] + s_red[1] + s_red[2] + s_red[3];
  const int r0 = s_bound[seg];
  const int n = s_bound[seg + 1] - r0;
  if (tid == 0 && seg < n_exp) offsets[seg] = dst;   // rank 0's segments start the experts
  if (tid == 0 && seg == 0) offsets[n_exp] = end;
  for (int i = tid; i < n; i += 256) {
    rows[dst + i] = r0 + i;
    pos[r0 + i] = dst + i;
  }
  for (int i = end + seg * 256 + tid; i < max_rows; i += gridDim.x * 256) pos[i] = -1;
}

hipError_t launch_merge_segments(const int32_t* counts, int S, int n_exp, int max_rows, int32_t* offsets,
                                 int32_t* rows, int32_t* pos, void* tail, int tail_bytes, hipStream_t s) {
  if (S < 1 || S > kMaxSeg || n_exp < 1 || S % n_exp != 0 || max_rows > (1 << 24))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(merge_segments_kernel, dim3(static_cast<unsigned>(S)), dim3(256), 0, s, counts, S, n_exp,
                     max_rows, offsets, rows, pos, static_cast<uint32_t*>(tail), tail_bytes / 4);
  return hipGetLastError();
}

}  // namespace eimoe
