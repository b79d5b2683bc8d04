// 3-D non-maximum suppression on gfx950 (replaces the reference's nms_3d_cuda,
// csrc/cuda/nms_3d_cuda.cu:49-162, bound as _C.nms_3d by csrc/nms_3d.h:27-44).
//
// Two ways to the same result: a list of the overlapping pairs (ops3d_nms3d_pairs, second half of
// this file; what _C.nms_3d calls first), and an n x n bit mask with a greedy pass over it
// (ops3d_nms3d), for boxes that overlap too much for the list, negative thresholds and more than
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
__global__ __launch_bounds__(kBoxesPerWord) void nms3d_mask_kernel(const float *boxes, int n, float thresh,
                                                                   uint64_t *mask, int words, uint64_t *nzb,
                                                                   int nzw) {
  const int cb = blockIdx.x, rb = blockIdx.y;
  if (cb < rb) return;
  __shared__ float cbox[kBoxesPerWord * 6];
  const int t = threadIdx.x;
  const int c0 = cb * kBoxesPerWord, r0 = rb * kBoxesPerWord;
  const int ncol = min(n - c0, kBoxesPerWord), nrow = min(n - r0, kBoxesPerWord);
  for (int i = t; i < ncol * 6; i += kBoxesPerWord) cbox[i] = boxes[(int64_t)c0 * 6 + i];
  __syncthreads();
  if (t >= nrow) return;
  float me[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) me[k] = boxes[(int64_t)(r0 + t) * 6 + k];
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
    const uint64_t rm = removed_l[blk];
    uint64_t cur = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(rm >> 32)) << 32) |
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)rm);
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
//   nms3d_resolve_kernel  the rounds and the kept boxes' indices
// Too many pairs for the list, or more rounds than the mask's greedy pass would take (long chains
// of boxes that each depend on the one before), are reported as *num_keep = -1: the caller then
// runs ops3d_nms3d, whose cost does not depend on the overlaps.
// Figures: at ops3d_nms3d_pairs.
constexpr int kLists = 16;                 // pair lists (a counter each: fewer adds per address); one
                                           // wave of the resolve kernel serves each
constexpr int kCounterStride = 32;         // counters 128 bytes apart
constexpr int kPairsPerBox = 64;           // list capacity: above it a round over the list in one
                                           // workgroup costs as much as the mask's greedy pass
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
                                                         int capacity, uint32_t *__restrict__ counters) {
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

// The rounds, in one workgroup: three bitmaps of the boxes (kept, removed, blocked) in LDS, a wave
// per list, which drops decided pairs by compacting its list in place.  At least the first
// undecided box is decided in every round.  Then the kept boxes' original indices in score order.
constexpr int kResolveThreads = 64 * kLists;
__global__ __launch_bounds__(kResolveThreads) void nms3d_resolve_kernel(uint2 *lists, int capacity,
                                                                        const uint32_t *counters, int n,
                                                                        int max_rounds, const int64_t *order,
                                                                        int64_t *keep, int32_t *num_keep) {
  extern __shared__ uint32_t bits_l[];
  __shared__ int more_l[3], part_l[kLists];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int words = (n + 31) / 32;
  uint32_t *kept = bits_l, *removed = bits_l + words, *blocked = bits_l + 2 * words;
  for (int w = t; w < words; w += kResolveThreads) {
    kept[w] = 0;
    removed[w] = (w + 1) * 32 > n ? ~0u << (n & 31) : 0u;   // past the last box
    blocked[w] = 0;
  }
  if (t < 3) more_l[t] = 0;
  __syncthreads();
  const uint32_t total = counters[wv * kCounterStride];
  if (total > (uint32_t)capacity && lane == 0) more_l[2] = 1;   // a list overflowed
  __syncthreads();
  if (more_l[2]) {
    if (t == 0) *num_keep = -1;
    return;
  }
  uint2 *list = lists + (int64_t)wv * capacity;
  int cnt = (int)total;
  for (int round = 0;; ++round) {
    constexpr int U = 8;   // pairs per lane in flight
    int left = 0;
    for (int e0 = 0; e0 < cnt; e0 += 64 * U) {
      uint2 p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 64 + lane;
        p[u] = e < cnt ? list[e] : make_uint2(0u, 0u);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t a = p[u].x, b = p[u].y, ab = 1u << (a & 31), bb = 1u << (b & 31);
        bool open = a != b && !(removed[a >> 5] & ab) && !(removed[b >> 5] & bb);
        if (open) {
          if (kept[a >> 5] & ab) {
            atomicOr(&removed[b >> 5], bb);
            open = false;
          } else {
            atomicOr(&blocked[b >> 5], bb);
          }
        }
        // the open pairs to the front: every position written was read in this batch or before
        const uint64_t m = __ballot(open);
        if (open) list[left + __builtin_popcountll(m & (((uint64_t)1 << lane) - 1))] = p[u];
        left += __builtin_popcountll(m);
      }
    }
    cnt = left;
    if (cnt && lane == 0) more_l[round & 1] = 1;
    __syncthreads();
    const int more = more_l[round & 1];
    for (int w = t; w < words; w += kResolveThreads) {
      kept[w] |= ~(removed[w] | blocked[w]);
      blocked[w] = 0;
    }
    if (t == 0) more_l[(round & 1) ^ 1] = 0;
    __syncthreads();
    if (!more) break;
    if (round + 1 >= max_rounds) {
      if (t == 0) *num_keep = -1;
      return;
    }
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
  size_t sorted, order, lists, counters, placed, extents, bounds, cells, slots, bytes;
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

}  // namespace ops3d_nms

using ops3d_nms::kMaxBoxes;

extern "C" {

size_t ops3d_nms3d_workspace_bytes(int n) {
  if (n <= 0) return 0;
  const size_t words = ((size_t)n + 63) / 64, nzw = (words + 63) / 64;
  return (size_t)n * (words + nzw) * sizeof(uint64_t);
}

int ops3d_nms3d(const float *boxes_sorted, const int64_t *order, int n, float iou_threshold, void *workspace,
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
  hipLaunchKernelGGL(ops3d_nms::fill_zero_u64_kernel, dim3((unsigned)((nz + 255) / 256 < 4096 ? (nz + 255) / 256 : 4096)), dim3(256),
                     0, st, nzb, nz);
  hipLaunchKernelGGL(ops3d_nms::nms3d_mask_kernel, dim3(words, words), dim3(64), 0, st, boxes_sorted, n,
                     iou_threshold, mask, words, nzb, nzw);
  hipLaunchKernelGGL(ops3d_nms::nms3d_reduce_kernel, dim3(1), dim3(ops3d_nms::kReduceThreads),
                     (size_t)words * sizeof(uint64_t), st, mask, nzb, n, words, nzw, order, keep, num_keep);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
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
  uint2 *lists = reinterpret_cast<uint2 *>(ws + lay.lists);
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
  // The mask's greedy pass takes about 3.7 us per 64 boxes, a round 2 to 3 us
  const int max_rounds = 64 + n / 128;
  const size_t lds = (size_t)((n + 31) / 32) * 3 * sizeof(uint32_t);
  hipLaunchKernelGGL(nms3d_resolve_kernel, dim3(1), dim3(kResolveThreads), lds, st, lists, lay.capacity, counters, n,
                     max_rounds, ord, keep, num_keep);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

}  // extern "C"
