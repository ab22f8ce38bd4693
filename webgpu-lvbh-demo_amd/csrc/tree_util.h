// tree_util.h -- device helpers and the level plan shared by the tree kernels.
#pragma once

#include "device_util.h"

namespace lbvh {

// bvh-up-pass.js:208-210: zero components move off the "unwritten" sentinel.
__device__ __forceinline__ void perturb(float mn[3], float mx[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (mn[c] == 0.0f) mn[c] = -1e-8f;
    if (mx[c] == 0.0f) mx[c] = 1e-8f;
  }
}

// Box merges of quiet values.  For fminf / fmaxf the compiler canonicalises
// every operand it cannot prove quiet (a v_max_f32 x, x, x each: six per
// merge of two boxes, on every step of a climb).  The boxes a climb merges
// are always quiet -- results of fminf / fmaxf, or canonicalised where a
// caller's array is loaded -- and on quiet operands the bare instructions
// give exactly fminf's and fmaxf's results (the other operand for a quiet
// NaN; -0 below +0, and perturb keeps exact zeros out of the boxes anyway).
__device__ __forceinline__ float qmin(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float qmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

__device__ __forceinline__ void tri_box(const int4 a, const int4 b,
                                        const int4 c, float mn[3],
                                        float mx[3]) {
  const float ax = __int_as_float(a.x), ay = __int_as_float(a.y),
              az = __int_as_float(a.z);
  const float bx = __int_as_float(b.x), by = __int_as_float(b.y),
              bz = __int_as_float(b.z);
  const float cx = __int_as_float(c.x), cy = __int_as_float(c.y),
              cz = __int_as_float(c.z);
  mn[0] = fminf(ax, fminf(bx, cx)); mx[0] = fmaxf(ax, fmaxf(bx, cx));
  mn[1] = fminf(ay, fminf(by, cy)); mx[1] = fmaxf(ay, fmaxf(by, cy));
  mn[2] = fminf(az, fminf(bz, cz)); mx[2] = fmaxf(az, fmaxf(bz, cz));
}

__device__ __forceinline__ int4 pack3(const float v[3], int w) {
  return make_int4(__float_as_int(v[0]), __float_as_int(v[1]),
                   __float_as_int(v[2]), w);
}

// Node of a single leaf (N = 1): the reference's lone thread finds parent
// slot 0, arrives first and writes only the l_* half (f_1 = 1).
__device__ __forceinline__ void write_single_leaf_node(int4 *nodes, const float mn[3],
                                       const float mx[3]) {
  nodes[0] = pack3(mn, -1);
  nodes[1] = pack3(mx, 1);
  nodes[2] = make_int4(0, 0, 0, 0);
  nodes[3] = make_int4(0, 0, 0, 0);
}

// The gather of a wave's triangles through the permutation has two forms: a
// lane loads its own 48-byte row in three instructions, each of them touching a
// line per lane, or three lanes load a row, 16 contiguous bytes each, and an
// instruction touches a third as many.  Where the leaves' triangles are scattered
// and still in a cache (batched meshes, up to 5M triangles) the lines an
// instruction touches set the gather's time and the second form is faster: 80M
// triangles in 2,048 random meshes 5,710 -> 5,480 us, 5M random ones 420 -> 409.
// Where neighbouring leaves share lines the first is (16M heightfield 1,052,
// 1,062 with the second; batches of 80M surface triangles 5,080 / 5,160), so a wave
// picks by its own leaves: scattered if of its pairs of neighbours fewer than a
// quarter come from nearby triangles.  The two branches cost a 1M heightfield
// 139.0 -> 139.7 us.  Every lane of the wave calls it.
__device__ __forceinline__ bool scattered_gather(uint32_t pi) {
  const uint32_t other = (uint32_t)__shfl_xor((int)pi, 1, 64);
  return __popcll(__ballot(max(pi, other) - min(pi, other) < 16u)) < 16;
}

// Triangles of the wave's leaves into stage (192 int4s of LDS) with 16
// contiguous bytes per lane, three lanes per triangle.  Every lane of the wave
// calls it, with a leaf's triangle.
__device__ __forceinline__ void gather_rows(const int4 *tri, uint32_t pi,
                                            uint32_t N, int4 *stage) {
  const int lane = threadIdx.x & 63;
  int4 v[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int e = j * 64 + lane;
    const uint32_t p = (uint32_t)__shfl((int)pi, e / 3, 64);
    v[j] = tri[3 * (size_t)(p < N ? p : 0u) + e % 3];
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) stage[j * 64 + lane] = v[j];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int kFrontierMax = kTreeFrontier;
// Level L-1 tiles per tile: kFanIn (up to 32 x 128 items, typically a few
// hundred; a round holds at least kForestItems - kFrontierMax new ones), or
// all of them, up to kFanInMax, in one last tile.  Depends only on the
// number of level L-1 tiles, so the host's level plan and the kernel agree.
constexpr int kFanIn = 32;
constexpr int kFanInMax = 64;
__host__ __device__ constexpr uint32_t fan_in(uint32_t prev_tiles) {
  return prev_tiles <= (uint32_t)kFanInMax ? (uint32_t)kFanInMax
                                           : (uint32_t)kFanIn;
}

__device__ __forceinline__ int delta_next(uint32_t a, uint32_t b, uint32_t i) {
  return (a != b) ? (int)__clz(a ^ b) : 32 + (int)__clz(i ^ (i + 1u));
}

}  // namespace lbvh
