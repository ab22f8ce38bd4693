// k_forest.hip -- agglomeration levels without climbs: the leaf tiles of all but
// the largest meshes, and every item level.
//
// Reference: scripts/bvh/kernels/radix-tree.js (WGSL :137-238) and
// bvh-up-pass.js (WGSL :200-280); the same nodes, items and level plan as
// k_tree.hip's k_leaves, which the largest meshes take.
//
// A small mesh's tree is a chain of latencies.  In k_leaves most of a tile's
// life is the climb, one dependent LDS exchange per tree level: 16,000 of
// 25,000 cycles for a tile of 1,024 leaves (11 us as a kernel; a tile here 4.5,
// a level of items 4.5 against 8-13).  Here a tile of kForestLeaves
// leaves (or up to kForestItems items) builds its nodes at once, a thread per
// gap:
//   * a gap's node spans up to the nearest gap with a smaller delta on either
//     side.  Lane u of each wave keeps the mask of the wave's 64 gaps whose
//     delta is below u, built from the deltas' six bit planes; a gap of delta
//     v reads the masks of v, its own wave's first, and the nearest set bits
//     are its bounds;
//   * the boxes of the node's two children are range unions: a wave's sparse
//     table of unions of 2^k elements answers each with two reads (or a few,
//     across waves).  It takes 24 bytes per entry, which is why the tiles are
//     small;
//   * nodes and elements whose parent gap has no node in the tile are its
//     frontier, ranked by the bits of their first elements.
#include "tree_util.h"

namespace lbvh {

constexpr int kForestLeaves = kForestTile;
constexpr int kForestItems = 512;

// A wave's sparse table: entry i of level k is the union of its elements [i, i
// + 2^k), for k <= kTop and those i whose range ends in the wave.  A level
// less than the wave needs (ranges past 2^(kTop + 1) take two lookups more)
// lets five leaf tiles share a CU's LDS, not four.
constexpr int kTop = 4;
__host__ __device__ constexpr int table_level(int k) { return 65 * k - (1 << k) + 1; }
constexpr int kTable = table_level(kTop + 1);

template <int T>
struct ForestLds {
  float4 a[T / 64][kTable + 1];  // min.xyz, max.x; the last one: the whole wave
  float2 b[T / 64][kTable + 1];  // max.yz
  uint64_t below[T / 64][64];  // [wave][u]: its gaps with a delta below u
  uint64_t node_bits[T / 64];  // gaps whose node is complete in the tile
  uint64_t root_bits[T / 64];  // first elements of the frontier
  uint64_t id_bits[T / 64];    // node ids made here (kStage)
  signed char dm[T + 4];       // deltas by position: dm[p] before element p
};

// LDS written by a wave for itself: its operations complete in issue order.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Lanes whose value is below v, from the values' bit planes (as k_rt_tiles).
__device__ __forceinline__ uint64_t planes_below(const uint64_t (&pl)[6],
                                                 int v) {
  uint64_t lt = 0, eq = ~0ull;
#pragma unroll
  for (int b = 5; b >= 0; --b) {
    const uint64_t vb = 0ull - (uint64_t)((v >> b) & 1);
    lt |= eq & vb & ~pl[b];
    eq &= ~(pl[b] ^ vb);
  }
  return lt;
}

struct Box {
  float mn[3], mx[3];
};
template <int T>
__device__ __forceinline__ void join(const ForestLds<T> &L, int w, int e, Box &x) {
  const float4 p = L.a[w][e];
  const float2 r = L.b[w][e];
  x.mn[0] = qmin(x.mn[0], p.x); x.mn[1] = qmin(x.mn[1], p.y);
  x.mn[2] = qmin(x.mn[2], p.z); x.mx[0] = qmax(x.mx[0], p.w);
  x.mx[1] = qmax(x.mx[1], r.x); x.mx[2] = qmax(x.mx[2], r.y);
}
template <int T>
__device__ __forceinline__ Box entry(const ForestLds<T> &L, int w, int e) {
  const float4 p = L.a[w][e];
  const float2 r = L.b[w][e];
  return {{p.x, p.y, p.z}, {p.w, r.x, r.y}};
}

// Joins wave w's elements [i, j] to x, entry i of the level that halves the
// range already in it.
__device__ __forceinline__ int range_level(int i, int j) {
  return min(kTop, 31 - __clz(j - i + 1));
}
template <int T>
__device__ __forceinline__ void join_rest(const ForestLds<T> &L, int w, int i,
                                          int j, int k, Box &x) {
  join(L, w, table_level(k) + j + 1 - (1 << k), x);
  if (j - i >= 2 << kTop) {
    join(L, w, table_level(kTop) + i + (1 << kTop), x);
    join(L, w, table_level(kTop) + j + 1 - (2 << kTop), x);
  }
}

// Union of elements [x, y].
template <int T>
__device__ __forceinline__ Box forest_box(const ForestLds<T> &L, int x, int y) {
  const int wx = x >> 6, wy = y >> 6;
  const int i = x & 63, j = wx == wy ? y & 63 : 63;
  const int k = range_level(i, j);
  Box r = entry(L, wx, table_level(k) + i);
  join_rest(L, wx, i, j, k, r);
  if (wx != wy) {
    const int t = y & 63, kt = range_level(0, t);
    join(L, wy, table_level(kt), r);
    join_rest(L, wy, 0, t, kt, r);
    for (int w = wx + 1; w < wy; ++w) join(L, w, kTable, r);
  }
  return r;
}

// The forest over m <= T elements.  Thread tid < m passes element tid: its
// box and the delta d of the gap after it (thread 0 also d0, the delta before
// element 0); range(e) gives any element's leaf range.  Writes the complete
// nodes.
// Threads whose element or gap is a frontier root return out with its first
// and last element, leaf range, box and outer deltas; rank is its place and
// count (every thread) the frontier's size.
struct ForestRoot {
  bool out;
  int l, r, dl, dr;
  float mn[3], mx[3];
  uint32_t rank, count;
};

template <int T, bool kStage, class Range>
__device__ __forceinline__ ForestRoot forest_round(
    ForestLds<T> &L, int m, const float mn[3], const float mx[3], int d,
    int d0, const Range &range, int N, int4 *nodes,
    int ts = 0) {
  constexpr int W = T / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool elem = tid < m;
  if (elem) L.dm[tid + 1] = (signed char)d;
  if (tid == 0) L.dm[0] = (signed char)d0;
  {
    // past the last gap: 63, below no value; a mesh's end (-1): below all
    const uint64_t ends = __ballot(elem && d < 0);
    const int v = elem && d >= 0 ? d : 63;
    uint64_t pl[6];
#pragma unroll
    for (int b = 0; b < 6; ++b) pl[b] = __ballot((v >> b) & 1);
    L.below[w][lane] = planes_below(pl, lane) | ends;
  }
  if (tid < W) L.root_bits[tid] = L.id_bits[tid] = 0ull;
  {
    Box x = {{mn[0], mn[1], mn[2]}, {mx[0], mx[1], mx[2]}};
    const auto put = [&](int e) {
      L.a[w][e] = make_float4(x.mn[0], x.mn[1], x.mn[2], x.mx[0]);
      L.b[w][e] = make_float2(x.mx[1], x.mx[2]);
      wave_lds_fence();
    };
    put(lane);
#pragma unroll
    for (int k = 0; k < kTop; ++k) {
      // lanes past the level repeat its last entry
      const int i = min(lane, 64 - (2 << k));
      x = entry(L, w, table_level(k) + i);
      join(L, w, table_level(k) + i + (1 << k), x);
      put(table_level(k + 1) + i);
    }
    join(L, w, table_level(kTop) + 16, x);  // lane 0: the whole wave
    join(L, w, table_level(kTop) + 32, x);
    join(L, w, table_level(kTop) + 48, x);
    if (lane == 0) put(kTable);
  }
  __syncthreads();
  // nearest smaller deltas: positions pl and pr (-1: none in the tile); the
  // gap after element 64 q + bit is position 64 q + bit + 1
  const bool gap = tid < m - 1;
  int pl = -1, pr = -1;
  if (gap) {
    const uint64_t mask = L.below[w][d];
    const uint64_t lo = mask & ((1ull << lane) - 1);
    const uint64_t hi = lane == 63 ? 0ull : mask & ~((2ull << lane) - 1);
    if (lo) pl = w * 64 + 64 - (int)__clzll((long long)lo);
    if (hi) pr = w * 64 + (int)__ffsll((unsigned long long)hi);
  }
  for (int q = w - 1; q >= 0 && __ballot(gap && pl < 0); --q) {
    const uint64_t mask = L.below[q][gap ? d : 0];
    if (gap && pl < 0 && mask) pl = q * 64 + 64 - (int)__clzll((long long)mask);
  }
  for (int q = w + 1; q * 64 < m && __ballot(gap && pr < 0); ++q) {
    const uint64_t mask = L.below[q][gap ? d : 0];
    if (gap && pr < 0 && mask) pr = q * 64 + (int)__ffsll((unsigned long long)mask);
  }
  if (gap && pl < 0 && L.dm[0] < d) pl = 0;
  const bool node = pl >= 0 && pr >= 0;
  const uint64_t made = __ballot(node);
  if (lane == 0) L.node_bits[w] = made;
  __syncthreads();
  const auto is_node = [&](int g) {
    return g >= 0 && g < m - 1 && (L.node_bits[g >> 6] >> (g & 63) & 1);
  };
  ForestRoot R;
  R.out = false;
  int first = 0, slot = 0;
  int4 quad[4];
  if (node) {
    const int x = pl, y = pr - 1;
    const int dl = L.dm[pl], dr = L.dm[pr];
    const Box lb = forest_box(L, x, tid), rb = forest_box(L, tid + 1, y);
    const int lo = range(x).x, s = range(tid).y, hi = range(y).y;
    const bool whole = lo == 0 && hi == N - 1;
    const int K = whole ? 0 : (dr > dl ? hi : lo);
    quad[0] = pack3(lb.mn, lo == s ? -(s + 1) : s);
    quad[1] = pack3(lb.mx, 2);
    quad[2] = pack3(rb.mn, hi == s + 1 ? -(s + 2) : s + 1);
    quad[3] = pack3(rb.mx, 0);
    slot = K - ts;
    if (kStage) {
      atomicOr(reinterpret_cast<unsigned long long *>(&L.id_bits[slot >> 6]),
               1ull << (slot & 63));
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) nodes[4 * (size_t)K + q] = quad[q];
    }
    if (!whole && !is_node(dr > dl ? pr - 1 : pl - 1)) {
      R.out = true;
      first = x;
      R.l = lo; R.r = hi; R.dl = dl; R.dr = dr;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        R.mn[c] = qmin(lb.mn[c], rb.mn[c]);
        R.mx[c] = qmax(lb.mx[c], rb.mx[c]);
      }
    }
  }
  if (elem && !R.out) {
    // an element on its own (one under a node here has that node's gap as
    // its parent's)
    const int2 e = range(tid);
    const int dl = L.dm[tid];
    if (!(e.x == 0 && e.y == N - 1) && !is_node(d > dl ? tid : tid - 1)) {
      R.out = true;
      first = tid;
      R.l = e.x; R.r = e.y; R.dl = dl; R.dr = d;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        R.mn[c] = mn[c];
        R.mx[c] = mx[c];
      }
    }
  }
  if (R.out)
    atomicOr(reinterpret_cast<unsigned long long *>(&L.root_bits[first >> 6]),
             1ull << (first & 63));
  __syncthreads();
  R.rank = R.count = 0;
#pragma unroll
  for (int q = 0; q < W; ++q) {
    const uint64_t bits = L.root_bits[q];
    R.count += (uint32_t)__popcll(bits);
    const int s = first >> 6;
    const uint64_t lower = q < s ? bits : (q == s ? bits & ((1ull << (first & 63)) - 1) : 0ull);
    R.rank += (uint32_t)__popcll(lower);
  }
  if (kStage) {
    // a leaf tile's node ids are its own positions: in id order through LDS
    // (the table is no longer read), four lanes per 64-byte node
    static_assert(!kStage || 4 * T <= W * (kTable + 1), "a quad per node");
    int4 *stage = reinterpret_cast<int4 *>(&L.a[0][0]);
    if (node) {
#pragma unroll
      for (int q = 0; q < 4; ++q) stage[4 * slot + q] = quad[q];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = j * T + tid, kk = e >> 2;
      if (L.id_bits[kk >> 6] >> (kk & 63) & 1)
        store_nt(nodes + 4 * (size_t)ts + e, stage[e]);
    }
  }
  return R;
}

// The round's frontier into the tile's slots (emit_frontier of k_tree.hip).
__device__ __forceinline__ void forest_emit(const ForestRoot &R, uint32_t tile,
                                            int4 *items_out,
                                            uint32_t *count_out, Ctl *ctl) {
  if (threadIdx.x == 0) {
    count_out[tile] = R.count;
    if (R.count > (uint32_t)kFrontierMax) atomicOr(&ctl->fault, kFaultFrontier);
  }
  if (R.out && R.rank < (uint32_t)kFrontierMax) {
    int4 *io = items_out + kItemInt4 * ((size_t)tile * kFrontierMax + R.rank);
    io[0] = make_int4(R.l, R.r, __float_as_int(R.mn[0]), __float_as_int(R.mn[1]));
    io[1] = make_int4(__float_as_int(R.mn[2]), __float_as_int(R.mx[0]),
                      __float_as_int(R.mx[1]), __float_as_int(R.mx[2]));
    io[2] = make_int4(R.dl, R.dr, 0, 0);
  }
}

// With segments (kSegs) every segment is a mesh of its own: positions, node ids
// and the permutation are relative to its first leaf.  Batches of 17,555
// triangles in 16 meshes 91 us with k_leaves / 81 here, of 713,000 in 300 152 /
// 143, of 4.8M in 700 456 / 448; of 18M in 1,000 it turns, 1,452 / 1,462.
//
// Level 0: kForestLeaves sorted leaves per block.  Gathers O_TRI and the leaf
// boxes as k_leaves does.  kStage: the nodes go out in id order through LDS,
// four lanes per node; a mesh of at most kForestDirect leaves, whose tiles are
// latency alone, stores them from the threads that made them (a build of 1,500
// 20.4 -> 19.7 us; one of 2^18 71.9 against 71.1 us staged, of 2^22 412
// against 380).
constexpr uint32_t kForestDirect = 1u << 17;
template <bool kStage, bool kSegs>
__global__ __launch_bounds__(kForestLeaves) void k_forest_leaves(
    const int4 *__restrict__ tri, const uint32_t *__restrict__ skeys,
    const int32_t *__restrict__ perm, uint32_t N, int4 *__restrict__ otri,
    int4 *__restrict__ items_out, uint32_t *__restrict__ count_out,
    int4 *nodes, Ctl *ctl, TreeSegs segs) {
  constexpr int T = kForestLeaves;
  __shared__ ForestLds<T> L;
  const int tid = threadIdx.x;
  const uint32_t gtile = xcd_tile(blockIdx.x, gridDim.x);
  uint32_t tile = gtile;
  if (kSegs) {  // the tile's mesh
    const uint32_t sg = segs.tile_seg[gtile];
    const uint32_t at = segs.seg_off[sg];
    tile -= segs.seg_tile0[sg];
    N = segs.seg_off[sg + 1] - at;
    tri += 3 * (size_t)at;
    skeys += at;
    perm += at;
    otri += 3 * (size_t)at;
    nodes += 4 * (size_t)at;
  }
  const int ts = (int)(tile * T);
  const int m = (int)min((uint32_t)T, N - (uint32_t)ts);
  const uint32_t k = (uint32_t)ts + tid;
  float mn[3] = {0.f, 0.f, 0.f}, mx[3] = {0.f, 0.f, 0.f};
  int d = -1, d0 = -1;
  // O_TRI goes out through LDS, each wave's 192 int4s through its own table
  static_assert(3 * 64 <= kTable, "a wave's triangles");
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  int4 *stage = reinterpret_cast<int4 *>(&L.a[w][0]);
  {
    const uint32_t kc = min(k, N - 1);  // a lane past the mesh: the last leaf
    const uint32_t pi = (uint32_t)perm[kc];
    const uint32_t k_here = skeys[kc];
    const uint32_t k_next = skeys[min(k + 1, N - 1)];
    const uint32_t k_0 = skeys[ts], k_prev = skeys[ts > 0 ? ts - 1 : 0];
    int4 a, b, c;
    if (scattered_gather(pi)) {
      gather_rows(tri, pi, N, stage);
      a = stage[3 * lane];
      b = stage[3 * lane + 1];
      c = stage[3 * lane + 2];
    } else if (tid < m) {
      const size_t src = 3 * (size_t)(pi < N ? pi : 0u);
      a = tri[src];
      b = tri[src + 1];
      c = tri[src + 2];
      stage[3 * lane] = a;
      stage[3 * lane + 1] = b;
      stage[3 * lane + 2] = c;
    }
    const int d_next = delta_next(k_here, k_next, k);
    const int d_prev = delta_next(k_prev, k_0, (uint32_t)(ts - 1));
    if (tid < m) {
      tri_box(a, b, c, mn, mx);
      perturb(mn, mx);
      d = k + 1 < N ? d_next : -1;
      d0 = ts > 0 ? d_prev : -1;
    }
  }
  wave_lds_fence();
  {
    int4 *o = otri + 3 * (size_t)(ts + 64 * w);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int e = j * 64 + lane;
      if (e < 3 * (m - 64 * w)) store_nt(o + e, stage[e]);
    }
  }
  wave_lds_fence();  // the table is written next
  if (N == 1) {
    if (tid == 0) {
      write_single_leaf_node(nodes, mn, mx);
      count_out[gtile] = 0u;
    }
    return;
  }
  if (k == N - 1) {
    const int4 z = make_int4(0, 0, 0, 0);
    int4 *last = nodes + 4 * (size_t)(N - 1);
    last[0] = z; last[1] = z; last[2] = z; last[3] = z;
  }
  const ForestRoot R = forest_round<T, kStage>(
      L, m, mn, mx, d, d0, [ts](int e) { return make_int2(ts + e, ts + e); },
      (int)N, nodes, ts);
  forest_emit(R, gtile, items_out, count_out, ctl);
}

// Levels >= 1: the frontiers of fan_in(prev_tiles) tiles of the level below,
// in rounds of at most kForestItems items (the previous round's frontier
// first, read back from the tile's own slots).
//
// What the levels replace: k_items, one thread per gap of up to 1,024 items with
// a sparse table of range minima for the bounds and a segment tree for the
// boxes, binary lifting over both: a 16M build 1,064 us with it, 1,048 here, 12M
// clustered 966 / 947, a build of 100,000 over leaf tiles of 1,024 62 / 51.
template <bool kSegs>
__global__ __launch_bounds__(kForestItems) void k_forest_items(
    uint32_t N, const int4 *__restrict__ items_in,
    const uint32_t *__restrict__ count_in, uint32_t prev_tiles,
    int4 *items_out,  // written, then read back
    uint32_t *__restrict__ count_out, int4 *nodes, Ctl *ctl, TreeSegs segs) {
  constexpr int T = kForestItems;
  __shared__ ForestLds<T> L;
  __shared__ int2 s_range[T];
  static_assert(kFanInMax <= 64 && kFrontierMax < T, "a lane per source tile");
  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t tile = blockIdx.x;
  uint32_t first = tile, prev0 = 0;  // its place in the mesh; source tile 0
  if (kSegs) {
    const uint32_t sg = segs.tile_seg[tile];
    const uint32_t at = segs.seg_off[sg];
    first -= segs.seg_tile0[sg];
    prev0 = segs.prev_tile0[sg];
    prev_tiles = segs.prev_tiles[sg];
    N = segs.seg_off[sg + 1] - at;
    nodes += 4 * (size_t)at;
  }
  const uint32_t fan = fan_in(prev_tiles);
  const uint32_t src0 = prev0 + first * fan;
  const uint32_t nsrc = min(fan, prev_tiles - first * fan);
  // every wave scans the source counts for itself: lane s, items up to and
  // with source s
  const uint32_t own = (uint32_t)lane < nsrc
                           ? min(count_in[src0 + lane], (uint32_t)kFrontierMax)
                           : 0u;
  const uint32_t upto = wave_scan_add(own);
  const int total = (int)__builtin_amdgcn_readlane((int)upto, 63);
  int taken = 0;  // source items used by earlier rounds
  int carry = 0;  // items of the previous round's frontier
  while (true) {
    const int fresh = min(total - taken, T - carry);
    const bool last = taken + fresh == total;
    const int m = carry + fresh;
    // the source of item g: the first with more than g items up to it
    const int g = taken + tid - carry;
    int s = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1)
      if ((int)__shfl(upto, s + step - 1, 64) <= g) s += step;
    const int before = (int)__shfl(upto - own, s, 64);
    float mn[3] = {0.f, 0.f, 0.f}, mx[3] = {0.f, 0.f, 0.f};
    int d = -1, d0 = -1;
    if (tid < m) {
      const int4 *src =
          tid < carry
              ? items_out + kItemInt4 * ((size_t)tile * kFrontierMax + tid)
              : items_in + kItemInt4 * ((size_t)(src0 + s) * kFrontierMax +
                                        (uint32_t)(g - before));
      const int4 a = src[0], b = src[1], c = src[2];
      s_range[tid] = make_int2(a.x, a.y);
      mn[0] = __int_as_float(a.z);
      mn[1] = __int_as_float(a.w);
      mn[2] = __int_as_float(b.x);
      mx[0] = __int_as_float(b.y);
      mx[1] = __int_as_float(b.z);
      mx[2] = __int_as_float(b.w);
      d0 = c.x;
      d = c.y;
    }
    const ForestRoot R = forest_round<T, false>(
        L, m, mn, mx, d, d0, [&](int e) { return s_range[e]; }, (int)N, nodes);
    forest_emit(R, tile, items_out, count_out, ctl);
    if (last) break;
    taken += fresh;
    carry = (int)min(R.count, (uint32_t)kFrontierMax);
    __syncthreads();  // the emitted items are visible to the whole block
  }
}

void launch_forest_leaves(uint32_t grid, const float4 *tri,
                          const uint32_t *skeys, const int32_t *perm,
                          uint32_t n, float4 *otri, int4 *items_out,
                          uint32_t *count_out, float4 *nodes, Ctl *ctl,
                          const TreeSegs &segs, hipStream_t s) {
  const bool direct = n <= kForestDirect;
  const auto leaves =
      segs.tile_seg
          ? (direct ? k_forest_leaves<false, true> : k_forest_leaves<true, true>)
          : (direct ? k_forest_leaves<false, false> : k_forest_leaves<true, false>);
  hipLaunchKernelGGL(leaves, dim3(grid), dim3(kForestLeaves), 0, s,
                     reinterpret_cast<const int4 *>(tri), skeys, perm, n,
                     reinterpret_cast<int4 *>(otri), items_out, count_out,
                     reinterpret_cast<int4 *>(nodes), ctl, segs);
}

void launch_items(uint32_t grid, uint32_t n, const int4 *items_in,
                  const uint32_t *count_in, uint32_t prev_tiles,
                  int4 *items_out, uint32_t *count_out, float4 *nodes, Ctl *ctl,
                  const TreeSegs &segs, hipStream_t s) {
  hipLaunchKernelGGL(
      segs.tile_seg ? k_forest_items<true> : k_forest_items<false>, dim3(grid),
      dim3(kForestItems), 0, s, n, items_in, count_in, prev_tiles, items_out,
      count_out, reinterpret_cast<int4 *>(nodes), ctl, segs);
}

}  // namespace lbvh
