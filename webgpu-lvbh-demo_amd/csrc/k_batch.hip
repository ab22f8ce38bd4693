// k_batch.hip -- per-mesh bounds and Morton keys of a batched build.
//
// A batched build treats S independent meshes, concatenated, in one set of
// launches.  Work is cut into sort tiles of SortSegs::items x kSortThreads
// triangles that never straddle a mesh; each block handles one tile.  The arithmetic is
// the single-mesh path's (aabb-z-idx.js:177-208), per mesh.
#include "device_util.h"

namespace lbvh {

// Per-mesh fp32 min/max of the vertices: a partial (min.xyz, max.xyz) per block,
// at most kBoundsBlocks a mesh, for k_batch_fold.  Also each triangle's box
// centre (3 x total floats: x, then y, then z).
__global__ __launch_bounds__(kSortThreads) void k_batch_bounds(
    const float4 *__restrict__ tri, const uint32_t *__restrict__ seg_off,
    BoundsBlocks blocks, float4 *__restrict__ partials,
    float *__restrict__ cen, uint32_t total) {
  static_assert(kSortThreads == kMapThreads, "TriChunks block size");
  __shared__ float4 s_tri[3 * kMapThreads];
  const uint32_t blk = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t sg = blocks.blk_seg[blk];
  const uint32_t blk0 = blocks.seg_blk0[sg];
  const uint32_t share = blocks.seg_blk0[sg + 1] - blk0;  // the mesh's blocks
  struct {
    uint32_t begin, end;
  } r;
  {
    const uint32_t s0 = seg_off[sg], s1 = seg_off[sg + 1];
    const uint32_t per = (s1 - s0 + share - 1) / share;
    r.begin = min(s0 + (blk - blk0) * per, s1);
    r.end = min(r.begin + per, s1);
  }
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
    partials[2 * blk] = make_float4(v[0], v[1], v[2], 0.0f);
    partials[2 * blk + 1] = make_float4(v[3], v[4], v[5], 0.0f);
  }
}

// Folds each mesh's partials, a wave per mesh, into the slot of its first block.
// (One set of accumulators per mesh, met by atomics, took a launch to clear too
// and the bounds of 64 meshes, 683,000 triangles, 15.3 us where these take 12.3.
// Folded by every Morton block instead, 80M triangles in 2,048 meshes take 20
// us more.)
__global__ __launch_bounds__(64) void k_batch_fold(
    const float4 *__restrict__ partials, const uint32_t *__restrict__ seg_blk0,
    float4 *__restrict__ folded) {
  const uint32_t b0 = seg_blk0[blockIdx.x], nb = seg_blk0[blockIdx.x + 1] - b0;
  if (nb == 0) return;  // an empty mesh
  constexpr uint32_t kPer = kBoundsBlocks / 64;
  float4 lo[kPer], hi[kPer];
#pragma unroll
  for (uint32_t q = 0; q < kPer; ++q) {
    if (q * 64 >= nb) break;
    const uint32_t b = b0 + min(q * 64 + threadIdx.x, nb - 1);
    lo[q] = partials[2 * b];
    hi[q] = partials[2 * b + 1];
  }
  float v[6] = {lo[0].x, lo[0].y, lo[0].z, hi[0].x, hi[0].y, hi[0].z};
#pragma unroll
  for (uint32_t q = 1; q < kPer; ++q) {
    if (q * 64 >= nb) break;
    v[0] = fminf(v[0], lo[q].x); v[1] = fminf(v[1], lo[q].y);
    v[2] = fminf(v[2], lo[q].z); v[3] = fmaxf(v[3], hi[q].x);
    v[4] = fmaxf(v[4], hi[q].y); v[5] = fmaxf(v[5], hi[q].z);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    v[c] = wave_min(v[c]);
    v[3 + c] = wave_max(v[3 + c]);
  }
  if (threadIdx.x == 0) {
    folded[2 * b0] = make_float4(v[0], v[1], v[2], 0.0f);
    folded[2 * b0 + 1] = make_float4(v[3], v[4], v[5], 0.0f);
  }
}

// Per-mesh leaf AABB centre -> Morton key, plus the first sort pass's
// per-tile digit counts (tile-major, cnt0[tile * R + d], as the batched
// sort keeps them).  Bounds: host-provided fp32
// (6 per mesh; centres from the triangles) or k_batch_fold's, with
// k_batch_bounds' centres (cen non-null).
template <int kBits, int kItems>
__global__ __launch_bounds__(kSortThreads) void k_batch_morton(
    const float4 *__restrict__ tri, const float *__restrict__ cen,
    uint32_t total, SortSegs segs, const float *__restrict__ seg_bounds,
    BoundsBlocks blocks, const float4 *__restrict__ folded, int div_mode,
    uint32_t *__restrict__ keys, uint32_t *__restrict__ cnt0) {
  constexpr int kR = 1 << kBits;
  __shared__ uint32_t s_hist[kR];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t sg = segs.tile_seg[tile];
  const TileRange r = sort_tile_range(tile, 0u, segs, kItems * kSortThreads);
  const uint32_t base = r.begin, end = r.end;
  for (int d = threadIdx.x; d < kR; d += kSortThreads) s_hist[d] = 0u;
  const float *lo = seg_bounds + 6 * sg, *hi = lo + 3;
  if (!seg_bounds) {
    lo = reinterpret_cast<const float *>(folded + 2 * blocks.seg_blk0[sg]);
    hi = lo + 4;
  }
  float bmin[3], ext[3], rcp[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    bmin[c] = lo[c];
    ext[c] = __fsub_rn(hi[c], lo[c]);
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
    // a part tile: its rows of kSortThreads keys, no more (10,000 meshes of ten
    // 31.2 us with every row of 16, 21.2 so)
    float ce[kItems][3];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (base + j * kSortThreads >= end) break;
      const uint32_t i = base + j * kSortThreads + threadIdx.x;
#pragma unroll
      for (int c = 0; c < 3; ++c)
        ce[j][c] = i < end ? __builtin_nontemporal_load(cen + c * cs + i) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (base + j * kSortThreads >= end) break;
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

void launch_batch_bounds(const float4 *tri, const uint32_t *seg_off,
                         const BoundsBlocks &blocks, uint32_t grid,
                         uint32_t num_segs, float4 *partials, float4 *folded,
                         float *cen, uint32_t total, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_bounds, dim3(grid), dim3(kSortThreads), 0, s, tri,
                     seg_off, blocks, partials, cen, total);
  hipLaunchKernelGGL(k_batch_fold, dim3(num_segs), dim3(64), 0, s, partials,
                     blocks.seg_blk0, folded);
}

void launch_batch_morton(const float4 *tri, const float *cen, uint32_t total,
                         const SortSegs &segs, uint32_t tiles,
                         const float *seg_bounds, const BoundsBlocks &blocks,
                         const float4 *folded, int div_mode, uint32_t *keys,
                         uint32_t *cnt0, int bits, hipStream_t s) {
#define LBVH_BATCH_MORTON(B, I)                                              \
  hipLaunchKernelGGL((k_batch_morton<B, I>), dim3(tiles), dim3(kSortThreads), \
                     0, s, tri, cen, total, segs, seg_bounds, blocks,        \
                     folded, div_mode, keys, cnt0)
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
