// k_raycast.hip -- closest-hit ray casting over the built BVH, following the
// demo path tracer's traversal, as a consumer check of the output layout.
//
// Reference: scripts/pathtracer/pathtracer.js intersect_bvh (:495-584),
// tri_intersect (Moller-Trumbore, :587-619), aabb_intersect (:621-628).
// Root = node 0; child < 0 is leaf -(child+1) in O_TRI; the nearer valid
// child is visited first and the other pushed.  Rays are 8 floats
// (origin.xyz, pad, dir.xyz, pad); hits are the path tracer's RayHit
// (normal.xyz, dist), dist = -1 for a miss.  Every operation is explicitly
// rounded so the CPU restatement in the oracle reproduces hits bit for bit.
#include "device_util.h"

namespace lbvh {

struct V3 {
  float x, y, z;
};

__device__ __forceinline__ V3 sub(V3 a, V3 b) {
  return {__fsub_rn(a.x, b.x), __fsub_rn(a.y, b.y), __fsub_rn(a.z, b.z)};
}
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
  return {__fsub_rn(__fmul_rn(a.y, b.z), __fmul_rn(a.z, b.y)),
          __fsub_rn(__fmul_rn(a.z, b.x), __fmul_rn(a.x, b.z)),
          __fsub_rn(__fmul_rn(a.x, b.y), __fmul_rn(a.y, b.x))};
}
__device__ __forceinline__ float dot(V3 a, V3 b) {
  return __fadd_rn(__fadd_rn(__fmul_rn(a.x, b.x), __fmul_rn(a.y, b.y)),
                   __fmul_rn(a.z, b.z));
}
__device__ __forceinline__ V3 v3(int4 v) {
  return {__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z)};
}

// The distance of tri_intersect (pathtracer.js:587-619), -1 for a miss; its early
// ends in one test.
__device__ __forceinline__ float tri_distance(V3 o, V3 d, V3 v0, V3 v1, V3 v2) {
  const V3 e1 = sub(v1, v0), e2 = sub(v2, v0);
  const V3 pvec = cross(d, e2);
  const float det = dot(e1, pvec);
  const float idet = __fdiv_rn(1.0f, det);
  const V3 tvec = sub(o, v0);
  const float u = __fmul_rn(dot(tvec, pvec), idet);
  const V3 qvec = cross(tvec, e1);
  const float v = __fmul_rn(dot(d, qvec), idet);
  const bool out = u < 0.f || u > 1.f || fabsf(det) < 1e-10f || v < 0.f || __fadd_rn(u, v) > 1.f;
  return out ? -1.f : __fmul_rn(dot(e2, qvec), idet);
}

// Its normal, taken once per ray for the closest hit.
__device__ __forceinline__ V3 tri_normal(V3 v0, V3 v1, V3 v2) {
  const V3 nrm = cross(sub(v1, v0), sub(v2, v0));
  // __builtin_sqrtf is correctly rounded (the default fp32 mode); HIP's
  // __fsqrt_rn maps to the hardware approximation, which is not.
  const float len = __builtin_sqrtf(dot(nrm, nrm));
  return {__fdiv_rn(nrm.x, len), __fdiv_rn(nrm.y, len), __fdiv_rn(nrm.z, len)};
}

// aabb_intersect (pathtracer.js:621-628): the entry distance t0, and whether
// the traversal takes the child (a -1e30 there is a miss).
__device__ __forceinline__ bool aabb_hit(V3 lo, V3 hi, V3 o, V3 inv, float dist,
                                         float &t0) {
  const float fx = __fmul_rn(__fsub_rn(hi.x, o.x), inv.x);
  const float fy = __fmul_rn(__fsub_rn(hi.y, o.y), inv.y);
  const float fz = __fmul_rn(__fsub_rn(hi.z, o.z), inv.z);
  const float nx = __fmul_rn(__fsub_rn(lo.x, o.x), inv.x);
  const float ny = __fmul_rn(__fsub_rn(lo.y, o.y), inv.y);
  const float nz = __fmul_rn(__fsub_rn(lo.z, o.z), inv.z);
  t0 = fmaxf(fminf(fx, nx), fmaxf(fminf(fy, ny), fminf(fz, nz)));
  const float t1 = fminf(fmaxf(fx, nx), fminf(fmaxf(fy, ny), fmaxf(fz, nz)));
  // (t0 is NaN only where t1 is)
  return t1 >= fmaxf(t0, 0.f) && t0 < dist && t0 != -1e30f;
}

constexpr int kRayStack = 64;  // the path tracer's is 32 (pathtracer.js:493)
constexpr int kRayLds = 24;    // entries of it in LDS; deeper ones are rare
constexpr int kRayThreads = 64;
constexpr uint32_t kRayChunk = 64;  // consecutive blocks on one XCD

// A step fetches one node or triangle and waits for it, and a frame lasts as
// long as its longest waves (those that cross dense clusters), so what counts
// is the latency of a step:
//   * one fetch for either kind: lanes at a node and lanes at a triangle wait
//     together, not one after the other;
//   * the stack's first kRayLds entries are in LDS (an array indexed per lane
//     is in scratch memory; 24 words per lane leave the CU its 24 waves), in
//     blocks of one wave, so a finished wave's share is free at once;
//   * the normal, a square root and three divisions, is taken once at the
//     end, of the closest hit;
//   * kRayChunk blocks (4,096 rays) in a row run on one XCD, whose L2 then
//     holds the nodes they share (1M rays of a frame over 1M triangles 398 ->
//     317 us).
//   * the stack's top is at hand when a step ends in a pop;
//   * a step is straight-line code: a branch costs a wave some 16 cycles and a
//     mask, so addresses are selected, the far child is stored above the top
//     whether it is pushed or not, the triangle test has no early ends, and
//     one branch holds all of the stack past LDS.
// Calls back to back in us, with a fetch per kind, blocks of 256 and the stack in
// scratch memory / now: a 512 x 512 frame over 100,000 clustered triangles 286 /
// 204, 1,024 x 1,024 over a heightfield of 300,000 261 / 152, 2^14 scattered rays over
// 4,097 uniform triangles 81 / 50, 1M over 1M uniform 1,615 / 1,110, over a surface of
// 300,000 647 / 550 (540 before the straight-line steps); 1M over 100 triangles lose,
// 75.4 / 77.4 (80 in blocks of 256): with the tree in L1 a step's instructions count,
// and a straight-line step has more.
// Dropping popped nodes beyond the closest hit lost (the stack entries
// double), and so did descending to a leaf per lane before any test, touching
// both children ahead, a step that takes a leaf together with the node that
// comes off the stack after it (the first frame 222 -> 244), and a higher
// priority for waves with many steps (235).
__global__ __launch_bounds__(kRayThreads) void k_raycast(
    const int4 *__restrict__ nodes, const int4 *__restrict__ tri, uint32_t n,
    const float4 *__restrict__ rays, uint32_t count, float4 *__restrict__ hits,
    uint32_t max_steps) {
  // entry k in row k + 1; row 0: of an empty stack; the last one: past them
  __shared__ int s_stack[kRayLds + 2][kRayThreads];
  int deep[kRayStack - kRayLds];
  const uint32_t tid = threadIdx.x;
  // chunks of kRayChunk blocks go to the XCDs in turn; the rest as they come
  constexpr uint32_t kTurn = kXcds * kRayChunk;
  uint32_t blk = blockIdx.x;
  if (blk < gridDim.x / kTurn * kTurn)
    blk = blk / kTurn * kTurn + blk % kXcds * kRayChunk + blk / kXcds % kRayChunk;
  const uint32_t q = blk * kRayThreads + tid;
  if (q >= count) return;
  const float4 ro = rays[2 * (size_t)q], rd = rays[2 * (size_t)q + 1];
  const V3 o = {ro.x, ro.y, ro.z};
  V3 d = {rd.x, rd.y, rd.z};
  // d += (abs(d) < 1e-5) * 1e-5  (pathtracer.js:502-503)
  if (fabsf(d.x) < 1e-5f) d.x = __fadd_rn(d.x, 1e-5f);
  if (fabsf(d.y) < 1e-5f) d.y = __fadd_rn(d.y, 1e-5f);
  if (fabsf(d.z) < 1e-5f) d.z = __fadd_rn(d.z, 1e-5f);
  const V3 inv = {__fdiv_rn(1.0f, d.x), __fdiv_rn(1.0f, d.y),
                  __fdiv_rn(1.0f, d.z)};
  float dist = 1e30f;
  uint32_t hit = 0;  // the closest hit's triangle (dist < 1e30)
  int sp = 0;        // entries on the stack; -1: the traversal is over
  int node = 0;
  for (uint32_t step = 0; sp >= 0 && step < max_steps; ++step) {
    const bool leaf = node < 0;
    const uint32_t id = (uint32_t)(leaf ? ~node : node);
    const bool in = id < n;
    const char *base = leaf ? reinterpret_cast<const char *>(tri)
                            : reinterpret_cast<const char *>(nodes);
    const char *at = base + (uint64_t)(in ? id : 0u) * (leaf ? 48u : 64u);
    const int4 *at4 = reinterpret_cast<const int4 *>(at);
    const int4 a = at4[0], b = at4[1], c = at4[2];
    const int4 e = *reinterpret_cast<const int4 *>(at + (leaf ? 32 : 48));
    // The stack's top, read from LDS while those loads are under way.  (Read
    // when it is popped, from LDS or scratch by its depth, it was one generic
    // load, which waits on the vector memory path.)
    const int row = min(sp, kRayLds);
    int top = s_stack[row][tid], far = 0;
    bool pop, push = false;
    if (leaf) {
      const float h = tri_distance(o, d, v3(a), v3(b), v3(c));
      const bool closer = in && h > 0.f && h < dist;
      dist = closer ? h : dist;
      hit = closer ? id : hit;
      pop = true;
    } else {
      float lt, rt;
      const bool lv = aabb_hit(v3(a), v3(b), o, inv, dist, lt);
      const bool rv = aabb_hit(v3(c), v3(e), o, inv, dist, rt);
      const bool left = lv && (!rv || lt < rt);  // the nearer child first
      far = left ? c.w : a.w;
      node = left ? a.w : c.w;
      s_stack[row + 1][tid] = far;  // above the top if not pushed
      push = in && lv && rv;
      pop = !in || !(lv || rv);
      sp = in ? sp : 0;
    }
    if (sp >= kRayLds) {
      if (push && sp < kRayStack) deep[sp - kRayLds] = far;
      if (pop && sp > kRayLds) top = deep[sp - 1 - kRayLds];
    }
    node = pop ? top : node;
    sp = pop ? sp - 1 : min(sp + (push ? 1 : 0), kRayStack);
  }
  // RayHit: normal facing the ray, dist -1 for a miss (pathtracer.js:572-583)
  V3 nrm = {0.f, 0.f, 0.f};
  if (dist < 1e30f) {
    const int4 *v = tri + 3 * (size_t)hit;
    nrm = tri_normal(v3(v[0]), v3(v[1]), v3(v[2]));
  }
  const float s = dot(d, {-nrm.x, -nrm.y, -nrm.z}) > 0.f ? 1.f : -1.f;
  hits[q] = make_float4(s * nrm.x, s * nrm.y, s * nrm.z,
                        dist == 1e30f ? -1.f : dist);
}

void launch_raycast(const void *nodes, const float *tri, uint32_t n,
                    const float *rays, uint32_t count, float *hits,
                    hipStream_t s) {
  const uint32_t blocks = (count + kRayThreads - 1) / kRayThreads;
  const uint64_t cap = 4ull * n + 256;
  hipLaunchKernelGGL(k_raycast, dim3(blocks ? blocks : 1), dim3(kRayThreads),
                     0, s, static_cast<const int4 *>(nodes),
                     reinterpret_cast<const int4 *>(tri), n,
                     reinterpret_cast<const float4 *>(rays), count,
                     reinterpret_cast<float4 *>(hits),
                     (uint32_t)(cap > 0xFFFFFFFFull ? 0xFFFFFFFFull : cap));
}

}  // namespace lbvh
