// 3-D non-maximum suppression on gfx950 (replaces the reference's nms_3d_cuda,
// csrc/cuda/nms_3d_cuda.cu:49-162, bound as _C.nms_3d by csrc/nms_3d.h:27-44).
//
// Two ways to the same result: a list of the overlapping pairs (ops3d_nms3d_pairs, second half of
// this file; what _C.nms_3d calls first), and an n x n bit mask with a greedy pass over it
// (ops3d_nms3d, ops3d_nms3d_after_pairs), for boxes that overlap too much for the list, negative thresholds and more than
// 2^18 boxes.
//
// The mask: boxes are (x1, y1, z1, x2, y2, z2) fp32, already sorted by decreasing score (the caller
// sorts, as the reference's host code does with torch).  Two kernels:
//   * nms3d_mask_kernel: for every pair of 64-box blocks (row block <= column block), one wave
//     compares its 64 row boxes against the 64 column boxes staged in LDS and writes one 64-bit
//     word per row box: bit i set when the row box's IoU with column box i (a later box) exceeds
//     the threshold.  64 boxes per word is the wave width: lane r owns row box r.  It also marks
//     which words of a row are nonzero, in a per-row bitmap (one bit per mask word, set by
//     atomic OR; cleared by a fill kernel first): boxes overlap only their neighbours, so a row
//     has few nonzero words.
//   * nms3d_reduce_kernel: the greedy pass on the GPU, one workgroup (the reference copies the
//     whole mask to the host and loops there).  Walking the sorted boxes in order, a box not yet
//     removed is kept and its mask row is OR-ed into the removed set -- only the row's nonzero
//     words, found from its bitmap.  It writes the kept boxes' original indices (order[i]) in
//     score order and their number; only that number has to reach the host (to size the
//     result).
// IoU (reference devIoU_3d, nms_3d_cuda.cu:36-47): intersection extents max(min - max, 0),
// volumes as products of extents, inter / (Sa + Sb - inter), each step rounded in fp32 (no
// contraction), so a CPU restatement in fp32 makes the same decisions.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/ops3d_nms3d.h"

namespace ops3d_nms {

constexpr int kBoxesPerWord = 64;   // one wave64 = one 64-bit mask word
// The greedy pass keeps one removed flag per box in LDS: 2^19 boxes = 64 KB (the mask is then
// 32 GB, quadratic in the boxes).
constexpr int kMaxBoxes = 1 << 19;

__device__ __forceinline__ float iou3d(const float *a, const float *b) {
#pragma clang fp contract(off)
  const float left = fmaxf(a[0], b[0]), right = fminf(a[3], b[3]);
  const float top = fmaxf(a[1], b[1]), bottom = fminf(a[4], b[4]);
  const float front = fmaxf(a[2], b[2]), back = fminf(a[5], b[5]);
  const float w = fmaxf(right - left, 0.f), h = fmaxf(bottom - top, 0.f), d = fmaxf(back - front, 0.f);
  const float inter = w * h * d;
  const float sa = (a[3] - a[0]) * (a[4] - a[1]) * (a[5] - a[2]);
  const float sb = (b[3] - b[0]) * (b[4] - b[1]) * (b[5] - b[2]);
  return inter / (sa + sb - inter);
}

// grid: (column blocks, row blocks); block: 64 threads.  Blocks below the diagonal exit: the
// greedy pass reads only words at or after a box's own block.
// Box i at boxes[i * stride].
__global__ __launch_bounds__(kBoxesPerWord) void nms3d_mask_kernel(const float *boxes, int stride, int n,
                                                                   float thresh, uint64_t *mask, int words,
                                                                   uint64_t *nzb, int nzw) {
  const int cb = blockIdx.x, rb = blockIdx.y;
  if (cb < rb) return;
  __shared__ float cbox[kBoxesPerWord * 6];
  const int t = threadIdx.x;
  const int c0 = cb * kBoxesPerWord, r0 = rb * kBoxesPerWord;
  const int ncol = min(n - c0, kBoxesPerWord), nrow = min(n - r0, kBoxesPerWord);
  for (int i = t; i < ncol * 6; i += kBoxesPerWord) cbox[i] = boxes[(int64_t)(c0 + i / 6) * stride + i % 6];
  __syncthreads();
  if (t >= nrow) return;
  float me[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) me[k] = boxes[(int64_t)(r0 + t) * stride + k];
  uint64_t bits = 0;
  const int start = cb == rb ? t + 1 : 0;   // only later boxes
  for (int i = start; i < ncol; ++i)
    if (iou3d(me, cbox + i * 6) > thresh) bits |= (uint64_t)1 << i;
  mask[(int64_t)(r0 + t) * words + cb] = bits;
  if (bits != 0 && cb > rb)   // off-diagonal nonzero word: mark it in the row's bitmap
    atomicOr(reinterpret_cast<unsigned long long *>(nzb + (int64_t)(r0 + t) * nzw + (cb >> 6)),
             1ull << (cb & 63));
}

__global__ __launch_bounds__(256) void fill_zero_u64_kernel(uint64_t *p, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0;
}

constexpr int kReduceThreads = 256;

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
  return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32) |
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
}

// One block of kReduceThreads; the removed flags (`words` 64-bit words) live in LDS.  Per
// 64-box block: every wave holds the block's 64 diagonal mask words (lane i: box i's), resolves
// which boxes survive serially from them (in scalar registers, unrolled and branch-free: a
// branchy loop that waited on each survivor's readlane cost 8 K cycles per block), wave 0
// writes the survivors'
// indices (lane i: box i, at its rank among them), and the survivors' rows are OR-ed into the
// removed words of later blocks: thread t serves row t % 64 and every 4th of its bitmap words
// (from the one holding word blk + 1: a row's bitmap marks only words after its own block),
// loading the nonzero mask words they name, up to 8 at a time, and adding them with LDS atomic
// OR.  The next block's diagonal words, original indices and first kPrefetch bitmap words per
// thread are loaded one block ahead, issued after the serial resolution, so a block waits for
// about one round of loads (its survivors' mask words).  Loading further ahead (two blocks, or
// the mask words of every row of the next block before its survivors are known) measured no
// better: the compiler's wait counts across the loop's back edge are conservative, so later
// loads are waited for early.
constexpr int kPrefetch = 8;   // bitmap words per thread loaded ahead (rows of up to 2^17 boxes)

__global__ __launch_bounds__(kReduceThreads) void nms3d_reduce_kernel(const uint64_t *mask, const uint64_t *nzb,
                                                                      int n, int words, int nzw,
                                                                      const int64_t *order, int64_t *keep,
                                                                      int32_t *num_keep) {
  extern __shared__ uint64_t removed_l[];
  const int t = threadIdx.x, lane = t & 63, slot = t >> 6;
  constexpr int kSlots = kReduceThreads / 64;
  for (int w = t; w < words; w += kReduceThreads) removed_l[w] = 0;
  __syncthreads();
  const auto diag_of = [&](int blk) {
    const int nb = min(n - blk * 64, 64);
    return lane < nb ? mask[(int64_t)(blk * 64 + lane) * words + blk] : (uint64_t)0;
  };
  const auto order_of = [&](int blk) {
    const int nb = min(n - blk * 64, 64);
    return lane < nb ? order[blk * 64 + lane] : (int64_t)0;
  };
  // bitmap word j of this thread for block blk: q = (blk + 1) / 64 + slot + kSlots * j
  const auto bitmap_of = [&](int blk, int j) {
    const int row = blk * 64 + lane, q = ((blk + 1) >> 6) + slot + kSlots * j;
    return row < n && q < nzw ? nzb[(int64_t)row * nzw + q] : (uint64_t)0;
  };
  uint64_t diag_n = diag_of(0);
  int64_t ord_n = order_of(0);
  uint64_t bm_n[kPrefetch];
#pragma unroll
  for (int j = 0; j < kPrefetch; ++j) bm_n[j] = bitmap_of(0, j);
  int kept = 0;
  for (int blk = 0; blk < words; ++blk) {
    const uint64_t diag = diag_n;
    const int64_t ord = ord_n;
    uint64_t bm[kPrefetch];
#pragma unroll
    for (int j = 0; j < kPrefetch; ++j) bm[j] = bm_n[j];
    const int nb = min(n - blk * 64, 64);
    // serial resolution in scalar registers, unrolled and branch-free: box i survives when no
    // kept box has removed it; a survivor removes the boxes its diagonal word marks
    uint64_t cur = uniform64(removed_l[blk]);
    if (nb < 64) cur |= ~(((uint64_t)1 << nb) - 1);   // boxes past n: never kept
    uint64_t km = 0;   // boxes of this block that survive
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const uint64_t alive = ((cur >> i) & 1) ^ 1;
      km |= alive << i;
      cur |= readlane64(diag, i) & (uint64_t)0 - alive;
    }
    // the next block's words, issued only now: a wait for this block's words placed after them
    // (loads complete in order) would wait for them too
    if (blk + 1 < words) {
      diag_n = diag_of(blk + 1);
      ord_n = order_of(blk + 1);
#pragma unroll
      for (int j = 0; j < kPrefetch; ++j) bm_n[j] = bitmap_of(blk + 1, j);
    }
    if (t < 64 && ((km >> lane) & 1)) {
      const int rank = __builtin_popcountll(km & (((uint64_t)1 << lane) - 1));
      keep[kept + rank] = ord;
    }
    kept += __builtin_popcountll(km);
    if ((km >> lane) & 1) {   // this thread's row survived: OR its nonzero later words in
      const int64_t row = (int64_t)blk * 64 + lane;
      const int q0 = ((blk + 1) >> 6) + slot;
      const auto add_row_words = [&](int q, uint64_t b) {
        while (b) {
          uint64_t v[8];
          int w[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {   // up to 8 loads in flight
            w[u] = b ? (q << 6) + __builtin_ctzll(b) : -1;
            b &= b - 1;
            v[u] = w[u] >= 0 ? mask[row * words + w[u]] : (uint64_t)0;
          }
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (v[u]) atomicOr(reinterpret_cast<unsigned long long *>(removed_l + w[u]), (unsigned long long)v[u]);
        }
      };
#pragma unroll
      for (int j = 0; j < kPrefetch; ++j) add_row_words(q0 + kSlots * j, bm[j]);
      for (int q = q0 + kSlots * kPrefetch; q < nzw; q += kSlots) add_row_words(q, nzb[row * nzw + q]);
    }
    __syncthreads();   // later blocks read the removed words written above
  }
  if (t == 0) *num_keep = kept;
}

// ---------------------------------------------------------------------------------------------
// Suppression over a pair list.  Boxes overlap only their neighbours, so instead of the n x n bit
// mask the pairs (a, b) of ranks a < b whose IoU exceeds the threshold are listed, and the greedy
// rule -- b is kept exactly when no kept a of a pair (a, b) exists -- is resolved for all boxes at
// once, in rounds: a pair whose a is kept removes b; a pair with a removed end is dropped; a box
// that no undecided box precedes in a pair is kept.  The result is the greedy pass's (its rule has
// one solution), and a round replaces up to n/64 dependent steps, each a round trip to memory.
//   nms3d_rank_kernel     small n: rank of every box by counting, boxes written in score order
//   nms3d_gather_kernel   larger n, order given: the boxes written in score order, centre bounds
//   nms3d_cell_kernel, nms3d_place_kernel, nms3d_extent_kernel
//                         larger n: boxes reordered by cell (counting sort over 16^3 cells in
//                         Morton order), so that blocks of 64 boxes are compact, and the blocks'
//                         extents
//   nms3d_pair_kernel     the pairs: block pairs (larger n: those whose extents meet) of 64 x 64
//                         boxes
//   nms3d_resolve_kernel  the rounds -- chains (boxes that each depend on the one before, where a
//                         round decides little) by blocks of 64 boxes instead -- and the kept
//                         boxes' indices
// Too many pairs for the list are reported as *num_keep = -1: the caller then runs the mask path, whose
// cost does not depend on the overlaps, on the boxes and the order made here (ops3d_nms3d_after_pairs).
// Figures: at ops3d_nms3d_pairs.
constexpr int kLists = 16;                 // pair lists (a counter each: fewer adds per address); one
                                           // wave of the resolve kernel serves each
constexpr int kCounterStride = 32;         // counters 128 bytes apart
constexpr int kPairsPerBox = 64;           // list capacity: two rounds over it cost less than half of
                                           // the mask's greedy pass
constexpr int kChainPairsPerBox = 32;      // above it chains cost the resolve kernel, one workgroup, as
                                           // much as the mask path or more
constexpr int kMaxPairBoxes = 1 << 18;     // three bitmaps of the boxes in 96 KB of LDS
constexpr int kMaxRankBoxes = 8192;        // ranks by counting (n^2 comparisons), keys in 32 KB of LDS
constexpr int kCells = 4096;               // 16^3
constexpr int kMaxGatherBlocks = kMaxPairBoxes / 256;

// A box in score order: x1, y1, z1, x2, y2, z2, its rank, unused.
struct __align__(32) Box {
  float v[6];
  int rank;
  int pad;
};

__device__ __forceinline__ Box no_box() {   // compares false with everything
  Box b;
#pragma unroll
  for (int k = 0; k < 6; ++k) b.v[k] = __int_as_float(0x7fc00000);
  b.rank = 0;
  b.pad = 0;
  return b;
}

// Order-preserving key of a score: torch.sort's descending order (NaN first, the zeros equal).
__device__ __forceinline__ uint32_t score_key(float s) {
  if (s != s) return 0xfffffffeu;
  if (s == 0.f) s = 0.f;
  const uint32_t u = (uint32_t)__float_as_int(s);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Rank of box i = boxes with a greater key, plus those with the same key before it.  A block ranks
// kRankBoxes boxes; thread (slice, box) counts over every kRankSlices-th key (the keys of all boxes
// in LDS).  n <= kMaxRankBoxes.
constexpr int kRankBoxes = 16, kRankSlices = 64;
__global__ __launch_bounds__(kRankBoxes *kRankSlices) void nms3d_rank_kernel(const float *boxes, int64_t bs, int64_t cs,
                                                                            const float *scores, int64_t ss, int n,
                                                                            Box *sorted, int64_t *order,
                                                                            uint32_t *counters) {
  __shared__ uint32_t key_l[kMaxRankBoxes];
  __shared__ int part_l[kRankBoxes];
  const int t = threadIdx.x, box = t % kRankBoxes, slice = t / kRankBoxes;
  for (int j = t; j < n; j += kRankBoxes * kRankSlices) key_l[j] = score_key(scores[j * ss]);
  if (t < kRankBoxes) part_l[t] = 0;
  if (blockIdx.x == 0) {
    if (t < kLists) counters[t * kCounterStride] = 0;
    if (t < 64) {   // the last block of 64 boxes is filled up
      const int r = n + t;
      if (r < (n + 63) / 64 * 64) sorted[r] = no_box();
    }
  }
  __syncthreads();
  const int i = blockIdx.x * kRankBoxes + box;
  if (i < n) {
    const uint32_t key = key_l[i];
    int c = 0;
    // keys are below 2^32 - 1, so key + 1 > key_i says key >= key_i
#pragma unroll 4
    for (int j = slice; j < n; j += kRankSlices) c += key_l[j] + (j < i ? 1u : 0u) > key ? 1 : 0;
    atomicAdd(&part_l[box], c);
  }
  __syncthreads();
  if (t < kRankBoxes && i < n) {
    const int r = part_l[t];
    Box b;
#pragma unroll
    for (int k = 0; k < 6; ++k) b.v[k] = boxes[i * bs + k * cs];
    b.rank = r;
    b.pad = 0;
    sorted[r] = b;
    order[r] = i;
  }
}

__device__ __forceinline__ float centre(const Box &b, int ax) { return 0.5f * b.v[ax] + 0.5f * b.v[3 + ax]; }

// Boxes in score order (order given), and per block the bounds of their finite centres.
__global__ __launch_bounds__(256) void nms3d_gather_kernel(const float *boxes, int64_t bs, int64_t cs,
                                                           const int64_t *order, int n, Box *sorted, float *bounds,
                                                           uint32_t *counters, uint32_t *cells) {
  __shared__ float red_l[6][256];
  const int t = threadIdx.x, r = blockIdx.x * 256 + t;
  for (int c = blockIdx.x * 256 + t; c < kCells; c += gridDim.x * 256) cells[c] = 0;
  if (blockIdx.x == 0 && t < kLists) counters[t * kCounterStride] = 0;
  Box b = no_box();
  if (r < n) {
    const int64_t i = order[r];
#pragma unroll
    for (int k = 0; k < 6; ++k) b.v[k] = boxes[i * bs + k * cs];
    b.rank = r;
    sorted[r] = b;
  }
#pragma unroll
  for (int ax = 0; ax < 3; ++ax) {
    const float c = centre(b, ax);
    const bool ok = fabsf(c) < 3.0e38f;   // not for NaN or infinities
    red_l[ax][t] = ok ? c : 3.0e38f;
    red_l[3 + ax][t] = ok ? c : -3.0e38f;
  }
  for (int s = 128; s > 0; s >>= 1) {
    __syncthreads();
    if (t < s)
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        red_l[ax][t] = fminf(red_l[ax][t], red_l[ax][t + s]);
        red_l[3 + ax][t] = fmaxf(red_l[3 + ax][t], red_l[3 + ax][t + s]);
      }
  }
  __syncthreads();
  if (t < 6) bounds[blockIdx.x * 6 + t] = red_l[t][0];
}

__device__ __forceinline__ uint32_t spread4(uint32_t v) {   // bits 0..3 to bits 0, 3, 6, 9
  return (v & 1u) | ((v & 2u) << 2) | ((v & 4u) << 4) | ((v & 8u) << 6);
}

// Cell of every box and its slot in the cell (any order inside a cell: the cells only decide which
// boxes share a block).  Slots are counted in LDS first, so a crowded cell costs one global add per
// block.
__global__ __launch_bounds__(1024) void nms3d_cell_kernel(const Box *sorted, int n, const float *bounds, int nbounds,
                                                          uint32_t *cells, uint32_t *slots) {
  __shared__ uint32_t hist_l[kCells];
  __shared__ int lo_l[3], hi_l[3];
  const int t = threadIdx.x, r = blockIdx.x * 1024 + t;
  for (int c = t; c < kCells; c += 1024) hist_l[c] = 0;
  const auto sortable = [](float f) {   // float order as int order
    const int v = __float_as_int(f);
    return v < 0 ? v ^ 0x7fffffff : v;
  };
  if (t < 3) {
    lo_l[t] = sortable(3.0e38f);
    hi_l[t] = sortable(-3.0e38f);
  }
  __syncthreads();
  for (int e = t; e < nbounds * 6; e += 1024) {
    const int k = e % 6;
    if (k < 3)
      atomicMin(&lo_l[k], sortable(bounds[e]));
    else
      atomicMax(&hi_l[k - 3], sortable(bounds[e]));
  }
  __syncthreads();
  uint32_t cell = 0, slot = 0;
  if (r < n) {
    const Box b = sorted[r];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      const int lv = lo_l[ax], hv = hi_l[ax];
      const float lo = __int_as_float(lv < 0 ? lv ^ 0x7fffffff : lv), hi = __int_as_float(hv < 0 ? hv ^ 0x7fffffff : hv);
      const float x = (centre(b, ax) - lo) * (16.f / (hi - lo));
      const float y = x > 0.f ? fminf(x, 15.f) : 0.f;   // 0 for NaN too
      cell |= spread4((uint32_t)(int)y) << ax;
    }
    slot = atomicAdd(&hist_l[cell], 1u);
  }
  __syncthreads();
  for (int c = t; c < kCells; c += 1024)
    if (hist_l[c]) hist_l[c] = atomicAdd(&cells[c], hist_l[c]);
  __syncthreads();
  if (r < n) slots[r] = (cell << 18) | (hist_l[cell] + slot);   // 12 and 18 bits: n <= 2^18
}

// Boxes into cell order: start of the box's cell (every block scans the counts) plus its slot.
__global__ __launch_bounds__(1024) void nms3d_place_kernel(const Box *sorted, int n, const uint32_t *cells,
                                                           const uint32_t *slots, Box *placed) {
  __shared__ uint32_t start_l[kCells], wave_l[16];
  const int t = threadIdx.x, lane = t & 63, r = blockIdx.x * 1024 + t;
  uint32_t c[4], sum = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    c[k] = cells[t * 4 + k];
    sum += c[k];
  }
  uint32_t inc = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t v = __shfl_up(inc, d);
    if (lane >= d) inc += v;
  }
  if (lane == 63) wave_l[t >> 6] = inc;
  __syncthreads();
  uint32_t at = inc - sum;
  for (int w = 0; w < (t >> 6); ++w) at += wave_l[w];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    start_l[t * 4 + k] = at;
    at += c[k];
  }
  __syncthreads();
  if (r < n) {
    const uint32_t s = slots[r];
    placed[start_l[s >> 18] + (s & 0x3ffffu)] = sorted[r];
  } else if (r < (n + 63) / 64 * 64) {
    placed[r] = no_box();
  }
}

// Extent of each block of 64 boxes: min of the lower corners, max of the upper ones (a NaN
// coordinate is skipped: its box has no IoU above any threshold).  One wave per block.
__global__ __launch_bounds__(256) void nms3d_extent_kernel(const Box *placed, int nblk, float *extents) {
  const int lane = threadIdx.x & 63, blk = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blk >= nblk) return;
  const Box b = placed[blk * 64 + lane];
  float e[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    e[k] = b.v[k] == b.v[k] ? b.v[k] : (k < 3 ? INFINITY : -INFINITY);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) e[k] = k < 3 ? fminf(e[k], __shfl_xor(e[k], d)) : fmaxf(e[k], __shfl_xor(e[k], d));
  }
  if (lane < 6) {
    float v = e[0];
#pragma unroll
    for (int k = 1; k < 6; ++k) v = lane == k ? e[k] : v;
    extents[blk * 6 + lane] = v;
  }
}

// Pairs of boxes with IoU above thresh >= 0.  A pair whose boxes do not overlap on every axis has
// intersection 0 and IoU 0 or NaN, not above thresh, so six comparisons settle nearly all of them (a
// NaN coordinate makes the IoU NaN, and the comparison false as well); the IoU itself -- iou3d, the
// mask kernel's -- is computed only where some lane's boxes overlap.
//   PLACED: a workgroup takes one block of 64 row boxes and 64 column blocks, its waves in turn the
//   column blocks whose extents meet the row block's.  Of the two blocks only the boxes that meet
//   the other block's extent count (about 13 of 64 each on the clustered boxes of the benchmark):
//   they are packed in LDS and the wave's lanes take their pairs.
//   otherwise: one pair of blocks; lane r holds row box r, each wave a quarter of the columns, which
//   come four at a time through scalar registers.
// Pairs are collected in LDS and appended to the kLists lists with one add per workgroup.  A wave whose
// buffer fills up writes it out, each time to its next list, and what is left at the end goes to one
// list only if it is no more than such a piece: a few crowded blocks (or a single one) fill all lists
// evenly, so the lists hold kPairsPerBox pairs per box together, wherever the pairs lie.
constexpr int kPairBuf = 256;
constexpr int kColumns = 4;   // column boxes in scalar registers at a time
template <bool PLACED>
__global__ __launch_bounds__(256) void nms3d_pair_kernel(const Box *__restrict__ boxes, int nblk, float thresh,
                                                         const float *__restrict__ extents, uint2 *__restrict__ lists,
                                                         int capacity, uint32_t *counters) {
  __shared__ uint2 buf_l[4][kPairBuf];
  __shared__ int cnt_l[4], base_l;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the block's first list, hashed (the pairs lie in blocks at regular distances: the diagonal), its
  // waves' 4 apart, moved on by one with every piece
  static_assert(kLists == 16, "the top four bits of the hash");
  const uint32_t first_list = (blockIdx.x * 0x9e3779b1u + blockIdx.y * 0x85ebca77u) >> 28;
  uint32_t piece = first_list + 4u * (uint32_t)wv;
  int rb, cb0;
  if (PLACED) {
    rb = blockIdx.y;
    cb0 = blockIdx.x * 64;
    if (cb0 + 63 < rb) return;
  } else {   // row blocks p and nblk - 1 - p together have nblk + 1 column blocks
    const int p = (int)blockIdx.x / (nblk + 1), k = (int)blockIdx.x - p * (nblk + 1);
    if (k < nblk - p) {
      rb = p;
      cb0 = p + k;
    } else {
      rb = nblk - 1 - p;
      if (rb == p) return;
      cb0 = rb + (k - (nblk - p));
    }
  }
  const Box me = boxes[rb * 64 + lane];
  int cnt = 0;
  bool full = false;
  const auto overlap = [](const float *a, const float *b) {
    return (a[0] < b[3]) & (b[0] < a[3]) & (a[1] < b[4]) & (b[1] < a[4]) & (a[2] < b[5]) & (b[2] < a[5]);
  };
  // the wave's buffer out (LDS operations of one wave are in order)
  const auto write_out = [&]() {
    const uint32_t list = piece++ % kLists;
    uint2 *out = lists + (int64_t)list * capacity;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(counters + list * kCounterStride, (uint32_t)cnt);
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    __builtin_amdgcn_wave_barrier();
    if (base > (uint32_t)capacity) full = true;   // the call falls back to the mask
    for (int e = lane; e < cnt; e += 64)
      if (base + (uint32_t)e < (uint32_t)capacity) out[base + e] = buf_l[wv][e];
    __builtin_amdgcn_wave_barrier();
    cnt = 0;
  };
  // adds the pairs (a, b) of the lanes in `near` whose IoU is above thresh
  const auto add_pairs = [&](const Box &a, const Box &b, bool near) {
    if (__ballot(near) == 0) return;
    const bool hit = near && iou3d(a.v, b.v) > thresh;
    const uint64_t m = __ballot(hit);
    if (m == 0) return;
    if (hit) {
      const int at = cnt + __builtin_popcountll(m & (((uint64_t)1 << lane) - 1));
      buf_l[wv][at] = make_uint2((uint32_t)min(a.rank, b.rank), (uint32_t)max(a.rank, b.rank));
    }
    cnt += __builtin_popcountll(m);
    if (cnt > kPairBuf - 64) write_out();
  };
  if constexpr (PLACED) {
    __shared__ Box row_l[4][64], col_l[4][64];
    float re[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) re[k] = extents[rb * 6 + k];
    // a list has overflowed: the call falls back to the mask whatever is found here
    const bool over = counters[first_list * kCounterStride] > (uint32_t)capacity;
    bool meet = false;
    if (cb0 + lane < nblk && cb0 + lane >= rb) {
      const float *ce = extents + (cb0 + lane) * 6;
      meet = re[0] < ce[3] && ce[0] < re[3] && re[1] < ce[4] && ce[1] < re[4] && re[2] < ce[5] && ce[2] < re[5];
    }
    uint64_t todo = __ballot(meet);
    // every fourth of them from the wv-th; a column block's boxes are loaded one turn ahead
    const auto skip = [&](int k) {
      for (; k > 0; --k) todo &= todo - 1;
    };
    skip(wv);
    Box next = me;
    if (todo) next = boxes[(cb0 + __builtin_ctzll(todo)) * 64 + lane];
    full = over;
    while (todo && !full) {
      const int cb = cb0 + __builtin_ctzll(todo);
      const Box col = next;
      skip(4);
      if (todo) next = boxes[(cb0 + __builtin_ctzll(todo)) * 64 + lane];
      // the boxes of either block that meet the other block's extent, packed
      const float *ce = extents + cb * 6;
      const bool rn = overlap(me.v, ce), cn = overlap(col.v, re);
      const uint64_t rm = __ballot(rn), cm = __ballot(cn), below = ((uint64_t)1 << lane) - 1;
      const int nr = __builtin_popcountll(rm), nc = __builtin_popcountll(cm);
      __builtin_amdgcn_wave_barrier();
      if (rn) row_l[wv][__builtin_popcountll(rm & below)] = me;
      if (cn) col_l[wv][__builtin_popcountll(cm & below)] = col;
      __builtin_amdgcn_wave_barrier();
      const float inv = 1.f / (float)nc;
      for (int p0 = 0; p0 < nr * nc && !full; p0 += 64) {
        const int p = p0 + lane;
        // p / nc: exact, p + 1/2 lies at least 1/(2 nc) >= 1/128 from a multiple of nc and the
        // rounding moves it by less than 64 * 2^-22
        const int i = (int)(((float)p + 0.5f) * inv), j = p - i * nc;
        const bool in = p < nr * nc;
        const Box a = row_l[wv][in ? i : 0], b = col_l[wv][in ? j : 0];
        add_pairs(a, b, in && overlap(a.v, b.v) && (cb != rb || a.rank < b.rank));
      }
    }
  } else {
    const Box *col = boxes + cb0 * 64 + wv * 16;
    for (int i0 = 0; i0 < 16 && !full; i0 += kColumns) {
      Box c[kColumns];
      bool near[kColumns], any = false;
#pragma unroll
      for (int u = 0; u < kColumns; ++u) c[u] = col[i0 + u];
#pragma unroll
      for (int u = 0; u < kColumns; ++u) any |= near[u] = overlap(me.v, c[u].v);
      if (__ballot(any) == 0) continue;
#pragma unroll
      for (int u = 0; u < kColumns; ++u) add_pairs(me, c[u], near[u] && (cb0 != rb || wv * 16 + i0 + u > lane));
    }
  }
  if (lane == 0) cnt_l[wv] = cnt;
  __syncthreads();
  const int all = cnt_l[0] + cnt_l[1] + cnt_l[2] + cnt_l[3];
  if (all > kPairBuf) {
    if (cnt > 0) write_out();
    return;
  }
  uint2 *out = lists + (int64_t)first_list * capacity;
  if (threadIdx.x == 0) base_l = all ? (int)atomicAdd(counters + first_list * kCounterStride, (uint32_t)all) : 0;
  __syncthreads();
  uint32_t base = (uint32_t)base_l;
  for (int w = 0; w < wv; ++w) base += (uint32_t)cnt_l[w];
  for (int e = lane; e < cnt; e += 64)
    if (base + (uint32_t)e < (uint32_t)capacity) out[base + e] = buf_l[wv][e];
}

// Sum over the wave, on lane 63.
__device__ __forceinline__ int wave_total(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);   // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, true);   // row_bcast 15, 31
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, true);
  return v;
}

// The pairs resolved, in one workgroup: three bitmaps of the boxes (kept, removed, blocked) in LDS.
//
// Rounds first: a wave per list, which drops decided pairs by compacting its list in place.  At least
// the first undecided box is decided in every round.  With scores that fall independently of position
// two rounds (they take turns: one finds boxes to keep, the next removes what those overlap) decide
// 70 % or more of the undecided boxes: 5 rounds for 4096 boxes of the benchmark, 7 for 50 001, 11 on a
// grid with 11 pairs per box.  Scores that follow position (boxes in a row, equal scores in raster
// order) make chains: two rounds decide at most 1 % and read the other pairs again, for as many rounds
// as the chain is long.  So when the last two rounds decided less than a quarter, and as many more as
// that lets expect would cost more than the block pass, or the rounds have cost that much already, the
// rest is left to the block pass.
//
// Block pass: the open pairs are sorted by the 64-box block of their first box (a counting sort in
// LDS), and the blocks taken in order.  The pairs inside a block give its 64 x 64 mask, one wave
// resolves it, and the other pairs of the boxes that survive remove boxes of later blocks.  Two
// barriers per block, its pairs loaded one block ahead; at most n / 64 steps, where a chain of n boxes
// takes n / 2 rounds.  Figures at ops3d_nms3d_pairs.
constexpr int kResolveThreads = 64 * kLists;
// Costs in units of a pair read by a round (about 0.5 ns): a round besides its pairs, rounds per
// inverse share of the boxes decided, the block pass, each of its blocks, each of its pairs.
constexpr float kRoundCost = 2048.f, kRoundsPerShare = 8.f, kPassCost = 16384.f, kBlockCost = 3072.f, kSortCost = 2.5f;
// Chains with many pairs cost more than the mask.  An eighth of the pairs tells them apart: of 1024
// pairs, spread over the lists, those whose first box it does not block are about 16 / m in clusters of
// m boxes that all overlap (and 17 % with independent scores at 40 pairs per box), but (7/8)^33 = 1 % where
// every box follows 33 that overlap it.
constexpr uint32_t kChainFirst = 48;
constexpr int kMarkPairs = 1024;   // of a list: fewer are not worth a loop of their own
__global__ __launch_bounds__(kResolveThreads) void nms3d_resolve_kernel(uint2 *lists, int capacity,
                                                                        const uint32_t *counters, uint2 *by_block, int n,
                                                                        const int64_t *order, int64_t *keep,
                                                                        int32_t *num_keep) {
  extern __shared__ uint32_t bits_l[];
  __shared__ uint32_t left_l[2], open_l[2], part_l[kLists], over_l;
  __shared__ uint32_t mask_l[2][64][2];
  __shared__ uint64_t gone_l;
  __shared__ uint32_t pairs_l;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int words = (n + 31) / 32;
  uint32_t *kept = bits_l, *removed = bits_l + words, *blocked = bits_l + 2 * words;
  for (int w = t; w < words; w += kResolveThreads) {
    kept[w] = 0;
    removed[w] = (w + 1) * 32 > n ? ~0u << (n & 31) : 0u;   // past the last box
    blocked[w] = 0;
  }
  if (t < 2) left_l[t] = open_l[t] = 0;
  if (t == 0) over_l = pairs_l = 0;
  __syncthreads();
  const uint32_t total = counters[wv * kCounterStride];
  if (total > (uint32_t)capacity && lane == 0) over_l = 1;   // a list overflowed
  if (lane == 0) atomicAdd(&pairs_l, min(total, (uint32_t)capacity));
  __syncthreads();
  if (over_l) {
    if (t == 0) *num_keep = -1;
    return;
  }
  const uint2 *list = lists + (int64_t)wv * capacity;
  uint2 *list_out = lists + (int64_t)wv * capacity;
  const int nblk = (n + 63) / 64;
  int cnt = (int)total;
  if (pairs_l > (uint32_t)n * kChainPairsPerBox) {   // many pairs: the mask if they are chains
    for (int e = lane; e < cnt / 8; e += 64) {
      const uint32_t b = list[8 * e + (5 * e & 7)].y;
      if (!(blocked[b >> 5] >> (b & 31) & 1u)) atomicOr(&blocked[b >> 5], 1u << (b & 31));
    }
    __syncthreads();
    const uint32_t a = cnt ? list[(uint64_t)lane * (uint32_t)cnt / 64].x : 0u;
    const uint64_t m = __ballot(cnt && !(blocked[a >> 5] >> (a & 31) & 1u));
    if (lane == 0) atomicAdd(&open_l[0], (uint32_t)__builtin_popcountll(m));
    __syncthreads();
    const uint32_t first = open_l[0];
    __syncthreads();
    if (first < kChainFirst) {
      if (t == 0) *num_keep = -1;
      return;
    }
    if (t == 0) open_l[0] = 0;   // settle() has a barrier before it adds to it
  }
  // undecided boxes that no undecided box precedes are kept; the pairs left in all lists and the
  // boxes left undecided
  uint32_t more = 0, open_boxes = 0;
  const auto settle = [&](int round) {
    if (cnt && lane == 0) atomicAdd(&left_l[round & 1], (uint32_t)cnt);
    __syncthreads();
    more = left_l[round & 1];
    int u = 0;
    for (int w = t; w < words; w += kResolveThreads) {
      const uint32_t open = blocked[w] & ~removed[w];
      kept[w] |= ~(removed[w] | open);
      blocked[w] = 0;
      u += __builtin_popcount(open);
    }
    if (more && __ballot(u != 0) != 0) {
      u = wave_total(u);
      if (lane == 63) atomicAdd(&open_l[round & 1], (uint32_t)u);
    }
    if (t == 0) left_l[(round & 1) ^ 1] = open_l[(round & 1) ^ 1] = 0;
    __syncthreads();
    open_boxes = open_l[round & 1];
  };
  const auto pass_cost = [&]() {
    return kPassCost + kBlockCost * fminf((float)nblk, (float)more) + kSortCost * (float)more;
  };
  float first_pass = 0.f, spent = 0.f, open2 = (float)n, open1 = (float)n;   // undecided two rounds ago and one
  bool chains = false;
  for (int round = 0;; ++round) {
    constexpr int U = 8;   // pairs per lane in flight
    int left = 0;
    // the first round of a long list: nothing is decided yet, every pair only blocks its second box
    const bool mark = round == 0 && cnt > kMarkPairs;
    for (int e0 = 0; mark && e0 < cnt; e0 += 64 * U) {
      uint32_t b[U];
      bool seen[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 64 + lane;
        b[u] = e < cnt ? list[e].y : ~0u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) seen[u] = b[u] == ~0u || (blocked[b[u] >> 5] >> (b[u] & 31) & 1u);
#pragma unroll
      for (int u = 0; u < U; ++u)   // (adds to one word wait for each other)
        if (!seen[u]) atomicOr(&blocked[b[u] >> 5], 1u << (b[u] & 31));
    }
    for (int e0 = 0; !mark && e0 < cnt; e0 += 64 * U) {
      uint2 p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 64 + lane;
        p[u] = e < cnt ? list[e] : make_uint2(0u, 0u);
      }
      // the batch's state first: a box that this batch itself removes is seen in the next round
      uint32_t gone[U], keep_a[U], seen[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (e0 + u * 64 >= cnt) break;
        const uint32_t a = p[u].x, b = p[u].y;
        gone[u] = (removed[a >> 5] >> (a & 31) | removed[b >> 5] >> (b & 31)) & 1u;
        keep_a[u] = kept[a >> 5] >> (a & 31) & 1u;
        seen[u] = blocked[b >> 5] >> (b & 31) & 1u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (e0 + u * 64 >= cnt) break;
        const uint32_t b = p[u].y, bb = 1u << (b & 31);
        bool open = p[u].x != b && !gone[u];
        if (open) {
          if (keep_a[u] || !seen[u]) atomicOr(keep_a[u] ? &removed[b >> 5] : &blocked[b >> 5], bb);
          open = !keep_a[u];
        }
        // the open pairs to the front: every position written was read in this batch or before
        const uint64_t m = __ballot(open);
        const int to = left + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (open && to != e0 + u * 64 + lane) list_out[to] = p[u];
        left += __builtin_popcountll(m);
      }
    }
    if (!mark) cnt = left;
    spent += kRoundCost + (float)more;
    settle(round);
    if (!more) break;
    if (round == 0) first_pass = pass_cost();
    const float share = (open2 - (float)open_boxes) / open2;   // decided by the last two rounds
    chains = round > 0 && (spent > first_pass ||
                           (share < 0.25f && kRoundCost * kRoundsPerShare + 2.f * (float)more > pass_cost() * share));
    if (chains) break;
    open2 = open1;
    open1 = (float)open_boxes;
  }
  if (chains) {
    // counting sort by block: counts, then the ends of the blocks' runs, in `blocked` (all 0 now)
    uint32_t *end = blocked;
    constexpr int U = 8;
    // one add for the lanes that share the first lane's block (a list's neighbours mostly do)
    const auto add = [&](uint32_t b, bool in) {
      const uint32_t b0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
      const uint64_t same = __ballot(in && b == b0);
      uint32_t at = 0;
      if (in && (b != b0 || lane == __builtin_ctzll(same)))
        at = atomicAdd(&end[b], b == b0 ? (uint32_t)__builtin_popcountll(same) : 1u);
      const uint32_t first = (uint32_t)__shfl((int)at, same ? __builtin_ctzll(same) : 0);
      return b == b0 ? first + (uint32_t)__builtin_popcountll(same & (((uint64_t)1 << lane) - 1)) : at;
    };
    for (int e0 = 0; e0 < cnt; e0 += 64 * U) {
      uint32_t b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 64 + lane;
        b[u] = e < cnt ? list[e].x >> 6 : 0u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) add(b[u], e0 + u * 64 + lane < cnt);
    }
    __syncthreads();
    uint32_t run = 0;
    for (int b0 = 0; b0 < nblk; b0 += kResolveThreads) {
      const int b = b0 + t;
      const uint32_t c = b < nblk ? end[b] : 0u;
      uint32_t inc = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t v = __shfl_up(inc, d);
        if (lane >= d) inc += v;
      }
      if (lane == 63) part_l[wv] = inc;
      __syncthreads();
      uint32_t before_b = run;
#pragma unroll
      for (int k = 0; k < kLists; ++k) {
        before_b += k < wv ? part_l[k] : 0u;
        run += part_l[k];
      }
      if (b < nblk) end[b] = before_b + inc - c;   // its start; the placing moves it to its end
      __syncthreads();
    }
    for (int e0 = 0; e0 < cnt; e0 += 64 * U) {
      uint2 p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 64 + lane;
        p[u] = e < cnt ? list[e] : make_uint2(0u, 0u);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = e0 + u * 64 + lane < cnt;
        const uint32_t at = add(p[u].x >> 6, in);
        if (in) by_block[at] = p[u];
      }
    }
    if (t < 128) mask_l[t >> 6][t & 63][0] = mask_l[t >> 6][t & 63][1] = 0u;
    __syncthreads();   // (the pairs placed above are read below by other waves of this workgroup)
    constexpr int V = 4;
    uint2 next[V];
    uint32_t at = 0;             // first pair of block `blk`
    int blk = 0;
    const auto seek = [&]() {    // to the next block with pairs (or past the last)
      while (blk < nblk && end[blk] == at) ++blk;
    };
    const auto load = [&](uint2(&p)[V], uint32_t stop) {
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const uint32_t e = at + u * kResolveThreads + t;
        p[u] = e < stop ? by_block[e] : make_uint2(~0u, ~0u);
      }
    };
    seek();
    if (blk < nblk) load(next, end[blk]);
    for (int turn = 0; blk < nblk; turn ^= 1) {
      const uint32_t base = (uint32_t)blk, stop = end[blk], rest = at + V * kResolveThreads + t;
      uint2 p[V];
#pragma unroll
      for (int u = 0; u < V; ++u) p[u] = next[u];
      const auto inside = [&](const uint2 &q) {
        if (q.y >> 6 == base) atomicOr(&mask_l[turn][q.x & 63][(q.y >> 5) & 1], 1u << (q.y & 31));
      };
#pragma unroll
      for (int u = 0; u < V; ++u) inside(p[u]);
      for (uint32_t e = rest; e < stop; e += kResolveThreads) inside(by_block[e]);
      __syncthreads();   // this block's mask, and the boxes that earlier blocks removed
      at = stop;
      ++blk;
      seek();
      if (blk < nblk) load(next, end[blk]);
      const uint32_t w = 2 * base;
      if (wv == 0) {   // lane i: the boxes that box i suppresses; survivors with such boxes one by one
        const uint64_t later = (uint64_t)mask_l[turn][lane][1] << 32 | mask_l[turn][lane][0];
        uint64_t cur = uniform64((uint64_t)(w + 1 < (uint32_t)words ? removed[w + 1] : ~0u) << 32 | removed[w]);
        uint64_t todo = __ballot(later != 0) & ~cur;
        while (todo) {
          const uint64_t m = readlane64(later, __builtin_ctzll(todo));
          todo &= todo - 1;
          todo &= ~m;
          cur |= m;
        }
        if (lane < 2 && w + lane < (uint32_t)words) removed[w + lane] = (uint32_t)(cur >> (32 * lane));
        if (lane == 0) gone_l = cur;
        mask_l[turn][lane][0] = mask_l[turn][lane][1] = 0u;   // next written after two more barriers
      }
      __syncthreads();
      const uint64_t gone = uniform64(gone_l);
      const auto outside = [&](const uint2 &q) {
        if (q.y != ~0u && q.y >> 6 != base && !((gone >> (q.x & 63)) & 1) && !(removed[q.y >> 5] >> (q.y & 31) & 1u))
          atomicOr(&removed[q.y >> 5], 1u << (q.y & 31));
      };
#pragma unroll
      for (int u = 0; u < V; ++u) outside(p[u]);
      for (uint32_t e = rest; e < stop; e += kResolveThreads) outside(by_block[e]);
    }
    __syncthreads();
    for (int w = t; w < words; w += kResolveThreads) kept[w] = ~removed[w];
    __syncthreads();
  }
  // kept boxes before each word (in `blocked`), then every box its place
  int run = 0;
  for (int w0 = 0; w0 < words; w0 += kResolveThreads) {
    const int w = w0 + t;
    const int c = w < words ? __builtin_popcount(kept[w]) : 0;
    int inc = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(inc, d);
      if (lane >= d) inc += v;
    }
    if (lane == 63) part_l[wv] = inc;
    __syncthreads();
    int before = run;
#pragma unroll
    for (int k = 0; k < kLists; ++k) {
      before += k < wv ? part_l[k] : 0;
      run += part_l[k];
    }
    if (w < words) blocked[w] = (uint32_t)(before + inc - c);
    __syncthreads();
  }
  constexpr int U = 8;
  for (int i0 = 0; i0 < n; i0 += kResolveThreads * U) {
    int64_t o[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * kResolveThreads + t;
      o[u] = i < n ? order[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * kResolveThreads + t;
      if (i < n && ((kept[i >> 5] >> (i & 31)) & 1u))
        keep[blocked[i >> 5] + __builtin_popcount(kept[i >> 5] & ((1u << (i & 31)) - 1u))] = o[u];
    }
  }
  if (t == 0) *num_keep = run;
}

// Workspace of the pair path.
struct PairLayout {
  size_t sorted, order, lists, by_block, counters, placed, extents, bounds, cells, slots, bytes;
  int capacity;
  explicit PairLayout(int n) {
    const size_t nblk = ((size_t)n + 63) / 64;
    size_t at = 0;
    const auto take = [&](size_t b) {
      const size_t o = at;
      at = (at + b + 255) & ~(size_t)255;
      return o;
    };
    capacity = (int)((size_t)n * kPairsPerBox / kLists + kPairBuf);
    sorted = take(nblk * 64 * sizeof(Box));
    counters = take(kLists * kCounterStride * 4);
    lists = take((size_t)kLists * capacity * sizeof(uint2));
    by_block = take((size_t)kLists * capacity * sizeof(uint2));
    order = take(n <= kMaxRankBoxes ? (size_t)n * 8 : 0);
    const bool big = n > kMaxRankBoxes;
    placed = take(big ? nblk * 64 * sizeof(Box) : 0);
    extents = take(big ? nblk * 6 * 4 : 0);
    bounds = take(big ? (size_t)kMaxGatherBlocks * 6 * 4 : 0);
    cells = take(big ? kCells * 4 : 0);
    slots = take(big ? (size_t)n * 4 : 0);
    bytes = at;
  }
};

// The mask and the greedy pass over it; box i (in score order) at boxes_sorted[i * stride].
int mask_path(const float *boxes_sorted, int stride, const int64_t *order, int n, float iou_threshold, void *workspace,
              size_t workspace_bytes, int64_t *keep, int32_t *num_keep, void *stream) {
  if (n < 0) return OPS3D_FDA_EINVAL;
  if (n == 0) return OPS3D_FDA_OK;
  if (!boxes_sorted || !order || !keep || !num_keep || !workspace) return OPS3D_FDA_EINVAL;
  if (n > kMaxBoxes) return OPS3D_FDA_EINVAL;
  if (workspace_bytes < ops3d_nms3d_workspace_bytes(n) || (reinterpret_cast<uintptr_t>(workspace) & 7u))
    return OPS3D_FDA_EINVAL;
  const int words = (n + 63) / 64, nzw = (words + 63) / 64;
  uint64_t *mask = static_cast<uint64_t *>(workspace);
  uint64_t *nzb = mask + (size_t)n * words;   // per-row bitmap of nonzero mask words
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t nz = (int64_t)n * nzw;
  hipLaunchKernelGGL(fill_zero_u64_kernel, dim3((unsigned)((nz + 255) / 256 < 4096 ? (nz + 255) / 256 : 4096)), dim3(256),
                     0, st, nzb, nz);
  hipLaunchKernelGGL(nms3d_mask_kernel, dim3(words, words), dim3(64), 0, st, boxes_sorted, stride, n, iou_threshold, mask,
                     words, nzb, nzw);
  hipLaunchKernelGGL(nms3d_reduce_kernel, dim3(1), dim3(kReduceThreads), (size_t)words * sizeof(uint64_t), st, mask, nzb,
                     n, words, nzw, order, keep, num_keep);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

}  // namespace ops3d_nms

extern "C" {

size_t ops3d_nms3d_workspace_bytes(int n) {
  if (n <= 0) return 0;
  const size_t words = ((size_t)n + 63) / 64, nzw = (words + 63) / 64;
  return (size_t)n * (words + nzw) * sizeof(uint64_t);
}

int ops3d_nms3d(const float *boxes_sorted, const int64_t *order, int n, float iou_threshold, void *workspace,
                size_t workspace_bytes, int64_t *keep, int32_t *num_keep, void *stream) {
  return ops3d_nms::mask_path(boxes_sorted, 6, order, n, iou_threshold, workspace, workspace_bytes, keep, num_keep,
                              stream);
}

size_t ops3d_nms3d_pairs_workspace_bytes(int n) {
  return n <= 0 || n > ops3d_nms::kMaxPairBoxes ? 0 : ops3d_nms::PairLayout(n).bytes;
}

int ops3d_nms3d_pairs_ranks(int n) { return n > 0 && n <= ops3d_nms::kMaxRankBoxes ? 1 : 0; }

// Lists instead of the mask.  Measured, whole nms_nd call on clustered boxes, threshold 0.3, one
// MI355X: 4096 boxes 281 -> 50 us (mask 24 and greedy kernel 194 us, torch's sort 23 and six copies
// of the boxes became rank 7, pair 10, resolve 12 us), 50 001 boxes 4260 -> 193 us (mask 1265 and
// greedy kernel 2895 us became gather 5, cell 6, place 5, extent 3, pair 62, resolve 38 us; torch's
// sort 55 us of both).  The pair kernel of the large call is bound by the comparisons of the block
// pairs that meet (6 % of all), the resolve kernel by its rounds' latency on one CU.  Up to
// kMaxRankBoxes the order is counted (n^2 comparisons, 7 us at 4096 against torch's sort, gather and
// copies, 40 us) and all block pairs are compared: the four launches that order the boxes by cell
// cost about 20 us, more than the comparisons they would save.
// Scores that follow position, whole call, this path / sort and mask path, us (rounds to the end, as
// the kernel did before it had the block pass, in brackets): a chain of 3000 boxes 148 / 195 (862);
// rows whose boxes overlap the next 10, 4096 boxes 207 / 280, 16 384 boxes 672 / 957 (24 550); the next
// 30, 4096 boxes 350 / 286, 16 384 boxes 985 / 979 (66 500), 65 536 boxes 4030 / 5330 (813 000); equal
// scores in raster order, 20^3 boxes 344 / 491 (2970), 30^3 boxes 1080 / 1740 (6750).  The same grid
// with random scores 149 / 550.  One workgroup spends 1.5 to 2.5 ns on a pair of a chain (a round or
// two, the sort and the block pass), so at 32 pairs per box it is level with the mask path; rows that
// overlap the next 40 are left to the mask: 4096 boxes 289 / 278 (the block pass 414), 16 384 1118 / 976,
// 65 536 5680 / 5310.  Independent scores, or alike ones inside clusters, take a few rounds at any
// length: clusters of 100 boxes that nearly all overlap (40 pairs per box), 4096 boxes 134 / 343, 8300
// 326 / 620, 50 000 1222 / 4514 (lists of 32 per box, and so the mask: 344, 722, 4626), with scores
// alike inside a cluster 151 / 304, 339 / 576, 1305 / 5107.
int ops3d_nms3d_pairs(const float *boxes, int64_t box_stride, int64_t coord_stride, const float *scores,
                      int64_t score_stride, const int64_t *order, int n, float iou_threshold, void *workspace,
                      size_t workspace_bytes, int64_t *keep, int32_t *num_keep, void *stream) {
  using namespace ops3d_nms;
  if (n < 0) return OPS3D_FDA_EINVAL;
  if (n == 0) return OPS3D_FDA_OK;
  if (!boxes || !keep || !num_keep || !workspace || n > kMaxPairBoxes || !(iou_threshold >= 0.f))
    return OPS3D_FDA_EINVAL;
  if (order ? n <= kMaxRankBoxes : (n > kMaxRankBoxes || !scores)) return OPS3D_FDA_EINVAL;
  const PairLayout lay(n);
  if (workspace_bytes < lay.bytes || (reinterpret_cast<uintptr_t>(workspace) & 31u)) return OPS3D_FDA_EINVAL;
  char *ws = static_cast<char *>(workspace);
  Box *sorted = reinterpret_cast<Box *>(ws + lay.sorted), *placed = reinterpret_cast<Box *>(ws + lay.placed);
  uint32_t *counters = reinterpret_cast<uint32_t *>(ws + lay.counters);
  uint2 *lists = reinterpret_cast<uint2 *>(ws + lay.lists), *by_block = reinterpret_cast<uint2 *>(ws + lay.by_block);
  float *extents = reinterpret_cast<float *>(ws + lay.extents), *bounds = reinterpret_cast<float *>(ws + lay.bounds);
  uint32_t *cells = reinterpret_cast<uint32_t *>(ws + lay.cells), *slots = reinterpret_cast<uint32_t *>(ws + lay.slots);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nblk = (n + 63) / 64;
  const int64_t *ord = order;
  if (!order) {
    int64_t *ranked = reinterpret_cast<int64_t *>(ws + lay.order);
    ord = ranked;
    hipLaunchKernelGGL(nms3d_rank_kernel, dim3((n + kRankBoxes - 1) / kRankBoxes), dim3(kRankBoxes * kRankSlices), 0, st,
                       boxes, box_stride, coord_stride, scores, score_stride, n, sorted, ranked, counters);
    hipLaunchKernelGGL((nms3d_pair_kernel<false>), dim3((nblk + 1) / 2 * (nblk + 1)), dim3(256), 0, st, sorted, nblk,
                       iou_threshold, static_cast<const float *>(nullptr), lists, lay.capacity, counters);
  } else {
    const int ng = (n + 255) / 256, nc = (n + 1023) / 1024;
    hipLaunchKernelGGL(nms3d_gather_kernel, dim3(ng), dim3(256), 0, st, boxes, box_stride, coord_stride, order, n,
                       sorted, bounds, counters, cells);
    hipLaunchKernelGGL(nms3d_cell_kernel, dim3(nc), dim3(1024), 0, st, sorted, n, bounds, ng, cells, slots);
    hipLaunchKernelGGL(nms3d_place_kernel, dim3(nc), dim3(1024), 0, st, sorted, n, cells, slots, placed);
    hipLaunchKernelGGL(nms3d_extent_kernel, dim3((nblk + 3) / 4), dim3(256), 0, st, placed, nblk, extents);
    hipLaunchKernelGGL((nms3d_pair_kernel<true>), dim3((nblk + 63) / 64, nblk), dim3(256), 0, st, placed, nblk,
                       iou_threshold, extents, lists, lay.capacity, counters);
  }
  const size_t lds = (size_t)((n + 31) / 32) * 3 * sizeof(uint32_t);
  hipLaunchKernelGGL(nms3d_resolve_kernel, dim3(1), dim3(kResolveThreads), lds, st, lists, lay.capacity, counters,
                     by_block, n, ord, keep, num_keep);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

// Calls whose pairs overflow the lists, us, this way / from the scores again (torch's sort, a gather
// and copies) / mask path alone: 300 boxes that all overlap 75 / 109 / 79, 3000 175 / 219 / 188, 9001
// 467 / 470 / 428 (the order is not made again, but torch made it before too); 4096 boxes in clusters
// of 150 236 / 286 / 246, 20 000 in clusters of 120 1130 / 1130 / 1026, in a row with the next 60 each
// 4096 276 / 325 / 285, 16 384 1036 / 1044 / 985.  What is left above the mask path alone is the pair
// kernel up to the overflow, the cells' passes and a second wait for the host.
int ops3d_nms3d_after_pairs(const void *pairs_workspace, size_t pairs_workspace_bytes, const int64_t *order, int n,
                            float iou_threshold, void *workspace, size_t workspace_bytes, int64_t *keep,
                            int32_t *num_keep, void *stream) {
  using namespace ops3d_nms;
  if (n < 0) return OPS3D_FDA_EINVAL;
  if (n == 0) return OPS3D_FDA_OK;
  if (!pairs_workspace || n > kMaxPairBoxes || (order ? n <= kMaxRankBoxes : n > kMaxRankBoxes)) return OPS3D_FDA_EINVAL;
  const PairLayout lay(n);
  if (pairs_workspace_bytes < lay.bytes || (reinterpret_cast<uintptr_t>(pairs_workspace) & 31u)) return OPS3D_FDA_EINVAL;
  const char *ws = static_cast<const char *>(pairs_workspace);
  static_assert(sizeof(Box) % sizeof(float) == 0 && offsetof(Box, v) == 0, "boxes as rows of floats");
  return mask_path(reinterpret_cast<const float *>(ws + lay.sorted), (int)(sizeof(Box) / sizeof(float)),
                   order ? order : reinterpret_cast<const int64_t *>(ws + lay.order), n, iou_threshold, workspace,
                   workspace_bytes, keep, num_keep, stream);
}

}  // extern "C"
