// k_batch.hip -- per-mesh bounds and Morton keys of a batched build.
//
// A batched build treats S independent meshes, concatenated, in one set of
// launches.  Work is cut into sort tiles of SortSegs::items x kSortThreads
// triangles that never straddle a mesh; each block handles one tile.  The arithmetic is
// the single-mesh path's (aabb-z-idx.js:177-208), per mesh.
#include "device_util.h"

namespace lbvh {

// Order-preserving u32 encoding of fp32, so unsigned atomicMin/atomicMax
// compute float min/max exactly.
__device__ __forceinline__ uint32_t f2ord(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}

// Resets the per-mesh bounds accumulators (when the GPU computes the
// bounds).
__global__ __launch_bounds__(kMapThreads) void k_batch_prologue(
    uint32_t *seg_ord, uint32_t num_segs, int init_bounds) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (init_bounds)
    for (uint64_t i = first; i < 8ull * num_segs; i += stride)
      seg_ord[i] = ((i & 7) < 3) ? 0xFFFFFFFFu : 0u;  // min slots, max slots
}

// Per-mesh fp32 min/max of the vertices, one sort tile per block, and each
// triangle's box centre (3 x total floats: x, then y, then z) for
// k_batch_morton.
__global__ __launch_bounds__(kSortThreads) void k_batch_bounds(
    const float4 *__restrict__ tri, SortSegs segs, uint32_t *seg_ord,
    float *__restrict__ cen, uint32_t total) {
  static_assert(kSortThreads == kMapThreads, "TriChunks block size");
  __shared__ float4 s_tri[3 * kMapThreads];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t sg = segs.tile_seg[tile];
  const TileRange r =
      sort_tile_range(tile, 0u, segs, (uint32_t)(segs.items * kSortThreads));
  float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  // chunks begin on whole waves of the centres' arrays, so that a wave's store
  // is whole lines (80M triangles 1,010 -> 908 us; 623 without the stores)
  const uint32_t c0 = r.begin & ~63u;
  const uint32_t nch = (r.end - c0 + kMapThreads - 1) / kMapThreads;
  TriChunks tc{tri, 3 * (size_t)r.end, {}};
  if (nch) tc.load(c0);
  for (uint32_t k = 0; k < nch; ++k) {
    tc.stage(s_tri);
    if (k + 1 < nch) tc.load(c0 + (k + 1) * kMapThreads);
    __syncthreads();
    const uint32_t i = c0 + k * kMapThreads + threadIdx.x;
    if (i >= r.begin && i < r.end) {
      float mn[3], mx[3];
      staged_box(s_tri, threadIdx.x, mn, mx);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        v[c] = fminf(v[c], mn[c]);
        v[3 + c] = fmaxf(v[3 + c], mx[c]);
        __builtin_nontemporal_store(__fmul_rn(__fadd_rn(mx[c], mn[c]), 0.5f),
                                    cen + (size_t)c * cen_stride(total) + i);
      }
    }
    __syncthreads();  // s_tri is refilled for the next chunk
  }
  block_minmax(v);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      atomicMin(&seg_ord[8 * sg + c], f2ord(v[c]));
      atomicMax(&seg_ord[8 * sg + 3 + c], f2ord(v[3 + c]));
    }
  }
}

// Per-mesh leaf AABB centre -> Morton key, plus the first sort pass's
// per-tile digit counts (tile-major, cnt0[tile * R + d], as the batched
// sort keeps them).  Bounds: host-provided fp32
// (6 per mesh; centres from the triangles) or the GPU accumulators (centres
// from k_batch_bounds, cen non-null).
template <int kBits, int kItems>
__global__ __launch_bounds__(kSortThreads) void k_batch_morton(
    const float4 *__restrict__ tri, const float *__restrict__ cen,
    uint32_t total, SortSegs segs, const float *__restrict__ seg_bounds,
    const uint32_t *__restrict__ seg_ord, int div_mode,
    uint32_t *__restrict__ keys, uint32_t *__restrict__ cnt0) {
  constexpr int kR = 1 << kBits;
  __shared__ uint32_t s_hist[kR];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t sg = segs.tile_seg[tile];
  const TileRange r = sort_tile_range(tile, 0u, segs, kItems * kSortThreads);
  const uint32_t base = r.begin, end = r.end;
  for (int d = threadIdx.x; d < kR; d += kSortThreads) s_hist[d] = 0u;
  float bmin[3], ext[3], rcp[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float lo, hi;
    if (seg_bounds) {
      lo = seg_bounds[6 * sg + c];
      hi = seg_bounds[6 * sg + 3 + c];
    } else {
      lo = ord2f(seg_ord[8 * sg + c]);
      hi = ord2f(seg_ord[8 * sg + 3 + c]);
    }
    bmin[c] = lo;
    ext[c] = __fsub_rn(hi, lo);
    rcp[c] = __fdiv_rn(1.0f, ext[c]);
  }
  __syncthreads();
  const bool ieee = (div_mode == 1);
  const auto put = [&](uint32_t i, const float ce[3]) {
    const uint32_t key = morton_key(ce, bmin, ext, rcp, ieee);
    __builtin_nontemporal_store(key, keys + i);
    digit_add(s_hist, key & (kR - 1));
  };
  const size_t cs = cen_stride(total);
  // all of the thread's centres are loaded before any is used, 16 bytes at a
  // time in a whole tile (80M triangles 313 us a chunk at a time, 279 so, 224
  // with the wide accesses)
  if (cen && end - base == kItems * kSortThreads) {
    Words4 c[3][kItems / 4];
#pragma unroll
    for (int g = 0; g < kItems / 4; ++g)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        c[k][g] = __builtin_nontemporal_load(
            reinterpret_cast<const Words4 *>(cen + k * cs + base) +
            g * kSortThreads + threadIdx.x);
#pragma unroll
    for (int g = 0; g < kItems / 4; ++g) {
      Words4 kq;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float ce[3] = {__uint_as_float(c[0][g][e]),
                             __uint_as_float(c[1][g][e]),
                             __uint_as_float(c[2][g][e])};
        kq[e] = morton_key(ce, bmin, ext, rcp, ieee);
        digit_add(s_hist, kq[e] & (kR - 1));
      }
      // plain: the waves' ends share lines
      reinterpret_cast<Words4 *>(keys + base)[g * kSortThreads + threadIdx.x] = kq;
    }
  } else if (cen) {
    float ce[kItems][3];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint32_t i = base + j * kSortThreads + threadIdx.x;
#pragma unroll
      for (int c = 0; c < 3; ++c)
        ce[j][c] = i < end ? __builtin_nontemporal_load(cen + c * cs + i) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint32_t i = base + j * kSortThreads + threadIdx.x;
      if (i < end) put(i, ce[j]);
    }
  } else {
    __shared__ float4 s_tri[3 * kMapThreads];
    const uint32_t nch = (end - base + kMapThreads - 1) / kMapThreads;
    TriChunks tc{tri, 3 * (size_t)end, {}};
    if (nch) tc.load(base);
    for (uint32_t ch = 0; ch < nch; ++ch) {
      const uint32_t i = base + ch * kMapThreads + threadIdx.x;
      float ce[3];
      tc.stage(s_tri);
      if (ch + 1 < nch) tc.load(base + (ch + 1) * kMapThreads);
      __syncthreads();
      if (i < end) {
        float mn[3], mx[3];
        staged_box(s_tri, threadIdx.x, mn, mx);
#pragma unroll
        for (int c = 0; c < 3; ++c)
          ce[c] = __fmul_rn(__fadd_rn(mx[c], mn[c]), 0.5f);
        put(i, ce);
      }
      __syncthreads();  // s_tri is refilled for the next chunk
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kR; d += kSortThreads)
    cnt0[(size_t)tile * kR + d] = s_hist[d];
}

void launch_batch_prologue(uint32_t *seg_ord, uint32_t num_segs,
                           bool init_bounds, Ctl *ctl, hipStream_t s) {
  const uint64_t words = 8ull * num_segs;
  uint32_t blocks = (uint32_t)((words + kMapThreads - 1) / kMapThreads);
  if (blocks > 1024) blocks = 1024;
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(k_batch_prologue, dim3(blocks), dim3(kMapThreads), 0, s,
                     seg_ord, num_segs, init_bounds ? 1 : 0);
}

void launch_batch_bounds(const float4 *tri, const SortSegs &segs,
                         uint32_t tiles, uint32_t *seg_ord, float *cen,
                         uint32_t total, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_bounds, dim3(tiles), dim3(kSortThreads), 0, s,
                     tri, segs, seg_ord, cen, total);
}

void launch_batch_morton(const float4 *tri, const float *cen, uint32_t total,
                         const SortSegs &segs, uint32_t tiles,
                         const float *seg_bounds, const uint32_t *seg_ord,
                         int div_mode, uint32_t *keys, uint32_t *cnt0,
                         int bits, hipStream_t s) {
#define LBVH_BATCH_MORTON(B, I)                                              \
  hipLaunchKernelGGL((k_batch_morton<B, I>), dim3(tiles), dim3(kSortThreads), \
                     0, s, tri, cen, total, segs, seg_bounds, seg_ord,       \
                     div_mode, keys, cnt0)
  const bool small = segs.items == kSmallSortItems;
  if (bits == kWideBits) {
    if (small) LBVH_BATCH_MORTON(kWideBits, kSmallSortItems);
    else LBVH_BATCH_MORTON(kWideBits, kSortItems);
  } else {
    if (small) LBVH_BATCH_MORTON(kRadixBits, kSmallSortItems);
    else LBVH_BATCH_MORTON(kRadixBits, kSortItems);
  }
#undef LBVH_BATCH_MORTON
}

}  // namespace lbvh
