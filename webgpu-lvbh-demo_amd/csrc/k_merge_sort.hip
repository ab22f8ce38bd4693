// k_merge_sort.hip -- stable sort of a small single mesh by LDS tile sorts
// and rank merges.
//
// Reference: scripts/bvh/kernels/radix-sort.js (:161-500); the stable
// permutation is unique, so this equals the radix passes of k_sort.hip.
//
// A small sort is a chain of short kernels, each of a few microseconds of
// latency whatever its size: keys and radix passes of 64K triangles took nine
// launches and 43 us.  Here they are two and 18 us:
//   k_tile_sort    a block sorts up to kMsTile keys in LDS (10-11 us; small
//                  sorts take smaller tiles, tile_log).  In a build
//                  it makes the keys itself, from the box centres or the
//                  triangles, so the Morton pass is this kernel too.
//   k_merge        merges groups of 8, 16 or 32 sorted runs: every key finds
//                  its rank in each other run of its group and moves there
//                  (7 us for 32 runs of 2,048).
// Ranks cost (runs - 1) searches per key, so it pays while the chip is far
// from full (kMergeSortMax, kMergeBuildMax).
#include <algorithm>
#include <utility>

#include "device_util.h"

namespace lbvh {

constexpr int kMsPer = 2;  // keys per thread: a pair starts the runs of two
constexpr int kMsWave = 64 * kMsPer;  // keys per wave

// Every kSample-th sorted key also goes to a compact array, which the merge
// rounds search first.
constexpr int kSampleLog = 5;
constexpr uint32_t kSample = 1u << kSampleLog;

// Where a tile's keys come from.
enum { kSrcKeys, kSrcCentres, kSrcTriangles, kSrcWholeMesh };

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}

// One merge round: runs of kLen become runs of 2 kLen, from s_key[cur] to
// s_key[cur ^ 1].  A key's new position is its own offset plus its rank in
// the sibling run (keys equal to it count when the sibling comes first, so
// equal keys keep their order).  Runs inside a wave need no block barrier: a
// wave's LDS operations complete in issue order.
template <int kLen, bool kFull, int kTile>
__device__ __forceinline__ void merge_round(uint32_t (*s_key)[kTile],
                                            uint16_t (*s_idx)[kTile],
                                            int &cur) {
  const uint32_t p0 = 2 * threadIdx.x;
  const uint32_t sib = (p0 ^ kLen) & ~(uint32_t)(kLen - 1);
  const bool second = (p0 & kLen) != 0;
  const uint32_t *key_in = s_key[cur];
  const uint2 k2 = *reinterpret_cast<const uint2 *>(key_in + p0);
  const uint32_t i2 = *reinterpret_cast<const uint32_t *>(s_idx[cur] + p0);
  const uint32_t key[2] = {k2.x, k2.y};
  uint32_t pos[2] = {sib, sib};
  // without full keys a key plus one does not wrap
  const auto below = [&](uint32_t v, uint32_t k) {
    return kFull ? (second ? v <= k : v < k) : v < k + (second ? 1u : 0u);
  };
#pragma unroll
  for (int h = kLen / 2; h > 0; h >>= 1)
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (below(key_in[pos[e] + h - 1], key[e])) pos[e] += h;
  cur ^= 1;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    if (below(key_in[pos[e]], key[e])) pos[e] += 1;
    // own offset in the run + rank in the sibling + start of the pair
    const uint32_t to =
        (p0 & ~(uint32_t)(2 * kLen - 1)) + ((p0 + e) & (kLen - 1)) + pos[e] - sib;
    s_key[cur][to] = key[e];
    s_idx[cur][to] = (uint16_t)(e ? i2 >> 16 : i2 & 0xFFFFu);
  }
  if (2 * kLen <= kMsWave) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

__device__ __forceinline__ void ms_box_centre(const float4 *__restrict__ t,
                                              float mn[3], float mx[3],
                                              float ce[3]) {
  staged_box(t, 0, mn, mx);
#pragma unroll
  for (int k = 0; k < 3; ++k) ce[k] = __fmul_rn(__fadd_rn(mx[k], mn[k]), 0.5f);
}

template <int kSrc, bool kFull, int kTile>
__global__ __launch_bounds__(kTile / kMsPer) void k_tile_sort(
    MergeKeys src, uint32_t n, uint32_t *keys_out,
    int32_t *__restrict__ idx_out, uint32_t *__restrict__ smp_out) {
  constexpr int kThreads = kTile / kMsPer;
  __shared__ __align__(16) uint32_t s_key[2][kTile];
  __shared__ __align__(16) uint16_t s_idx[2][kTile];
  __shared__ float s_b[8];
  // past every key in order: real keys with this value come before
  constexpr uint32_t kPast = kFull ? 0xFFFFFFFFu : 0x7FFFFFFFu;
  const uint32_t tid = threadIdx.x;
  const uint32_t base = xcd_tile(blockIdx.x, gridDim.x) * (uint32_t)kTile;
  const uint32_t valid = min(n - base, (uint32_t)kTile);
  const uint32_t p0 = 2 * tid, i0 = base + p0;
  uint32_t key[2] = {kPast, kPast};
  if (kSrc == kSrcKeys) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (p0 + e < valid) key[e] = src.keys[i0 + e];
  } else {
    float ce[2][3];
    float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (kSrc == kSrcCentres) {
      // pairs are in the centre arrays' padding at worst
      const size_t cs = cen_stride(n);
      if (p0 < valid) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const float2 c = *reinterpret_cast<const float2 *>(src.cen + k * cs + i0);
          ce[0][k] = c.x;
          ce[1][k] = c.y;
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (p0 + e >= valid) continue;
        float mn[3], mx[3];
        ms_box_centre(src.tri + 3 * (size_t)(i0 + e), mn, mx, ce[e]);
        if (kSrc == kSrcWholeMesh) {
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            v[k] = fminf(v[k], mn[k]);
            v[3 + k] = fmaxf(v[3 + k], mx[k]);
          }
        }
      }
    }
    float bmin[3], ext[3], rcp[3];
    if (kSrc == kSrcTriangles) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        bmin[k] = src.p.bmin[k];
        ext[k] = src.p.ext[k];
        rcp[k] = src.p.rcp[k];
      }
    } else {
      if (kSrc == kSrcWholeMesh) {
        block_minmax(v);
        if (tid == 0)
          for (int k = 0; k < 6; ++k) s_b[k] = v[k];
      } else {
        // a wave folds a component of the partials, kFoldPer loads in flight
        for (uint32_t c = tid >> 6; c < 6; c += kThreads / 64) {
          constexpr uint32_t kFoldPer = kBoundsBlocks / 64;
          const float *part = reinterpret_cast<const float *>(src.partials) +
                              (c < 3 ? c : c + 1);
          const float sign = c < 3 ? 1.f : -1.f;  // max as a min
          float x[kFoldPer], b = INFINITY;
#pragma unroll
          for (uint32_t q = 0; q < kFoldPer; ++q)
            x[q] = part[8 * (size_t)min(q * 64 + (tid & 63), src.parts - 1)];
#pragma unroll
          for (uint32_t q = 0; q < kFoldPer; ++q) b = fminf(b, sign * x[q]);
          b = sign * wave_min(b);
          if ((tid & 63) == 0) s_b[c] = b;
        }
      }
      __syncthreads();
      // lane k divides for axis k
      const int axis = min((int)(tid & 63), 2);
      const float e = __fsub_rn(s_b[3 + axis], s_b[axis]);
      const float r = __fdiv_rn(1.0f, e);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        bmin[k] = s_b[k];
        ext[k] = __uint_as_float(lane_value(__float_as_uint(e), k));
        rcp[k] = __uint_as_float(lane_value(__float_as_uint(r), k));
      }
    }
    const bool ieee = src.p.div_mode == 1;
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (p0 + e < valid) key[e] = morton_key(ce[e], bmin, ext, rcp, ieee);
  }
  // runs of two, then rounds of merges while more than one run holds keys
  const bool swap = key[1] < key[0];
  int cur = 0;
  *reinterpret_cast<uint2 *>(s_key[0] + p0) =
      swap ? make_uint2(key[1], key[0]) : make_uint2(key[0], key[1]);
  *reinterpret_cast<uint32_t *>(s_idx[0] + p0) =
      swap ? (p0 << 16) | (p0 + 1) : ((p0 + 1) << 16) | p0;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#define LBVH_ROUND(L) merge_round<L, kFull, kTile>(s_key, s_idx, cur)
  LBVH_ROUND(2);
  LBVH_ROUND(4);
  LBVH_ROUND(8);
  LBVH_ROUND(16);
  LBVH_ROUND(32);
  LBVH_ROUND(64);
  __syncthreads();
  if (valid > 128) LBVH_ROUND(128);
  if (valid > 256) LBVH_ROUND(256);
  if (kTile > 512 && valid > 512) LBVH_ROUND(512 % kTile);
  if (kTile > 1024 && valid > 1024) LBVH_ROUND(1024 % kTile);
#undef LBVH_ROUND
  static_assert(kTile >= 512 && kTile <= 2048 && kMsWave == 128,
                "the rounds above");
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const uint32_t p = e * kThreads + tid;
    if (p < valid) {
      const uint32_t k = s_key[cur][p];
      keys_out[base + p] = k;
      idx_out[base + p] = (int32_t)(base + s_idx[cur][p]);
      if ((p & (kSample - 1)) == kSample - 1)
        smp_out[(base + p) >> kSampleLog] = k;
    }
  }
}

// x sorts before key k (equal: only when x's run comes first, le).
template <bool kFull>
__device__ __forceinline__ bool sorts_below(uint32_t x, uint32_t k, bool le) {
  // without full keys a key plus one does not wrap
  return kFull ? (le ? x <= k : x < k) : x < k + (le ? 1u : 0u);
}
// One merge round: merges groups of kWaves x kPer runs of 2^run_log keys (the
// last run and group may be short).  A block's waves take the same 64
// consecutive keys of a run and kPer runs of its group each, and add their
// ranks up.
//
// The ranks of the 64 keys in a run lie in a window that the first and the
// last of them bound to within kSample keys: their ranks among the run's
// samples, which a wave reads 64 at a time (in a long run every 2^x-th sample
// and then those between two).  A window of at most kWindow - 1 keys goes to
// LDS, where the runs' binary searches go side by side with constant steps:
// what bounds the kernel is instructions, about 45 per run and wave, so
// windows of exact size, searched in fewer but computed steps, took twice as
// long, as did whole tiles in LDS (L2 bandwidth).  Wider windows, where the
// runs' keys are spread unevenly, are searched in place.
// Between evenly spread runs a window holds 64 + 31 keys on average, with a
// deviation near 17: at 128 a fifth of the waves of 8 runs met a wider one.
constexpr int kWindow = 192;
constexpr int kSteps = 8;  // 2^kSteps > kWindow; reads past it decide nothing
constexpr int kMaxRunLog = kMsTileLog + 6;  // two readings of 64 samples

// Lanes whose x sorts before k (equal ones too when le), of the first c.
template <bool kFull>
__device__ __forceinline__ uint32_t count_below(uint32_t x, uint32_t k, bool le,
                                                uint32_t c) {
  const uint64_t first = c >= 64 ? ~0ull : (1ull << c) - 1;
  return (uint32_t)__popcll(__ballot(sorts_below<kFull>(x, k, le)) & first);
}

template <int kWaves, int kPer, bool kFull>
__global__ __launch_bounds__(64 * kWaves) void k_merge(
    const uint32_t *__restrict__ keys_in, const int32_t *__restrict__ idx_in,
    const uint32_t *__restrict__ smp_in, uint32_t *__restrict__ keys_out,
    int32_t *__restrict__ idx_out, uint32_t *__restrict__ smp_out, uint32_t n,
    int run_log) {
  constexpr uint32_t kRuns = kWaves * kPer;
  __shared__ uint32_t s_win[kWaves][kPer * kWindow + (1 << kSteps) - kWindow];
  __shared__ uint32_t s_rank[kWaves][64];
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t c0 = xcd_tile(blockIdx.x, gridDim.x) * 64;
  const uint32_t i = c0 + lane;
  const uint32_t run = c0 >> run_log;  // the chunk's run: lengths are
  const uint32_t g0 = run & ~(kRuns - 1);  // multiples of 64
  const uint32_t s0 = g0 + wave * kPer;    // this wave's runs
  uint32_t rank = 0, key = 0;
  int32_t val = 0;
  if (c0 < n) {
    const uint32_t at = min(i, n - 1);  // past the end: the last key again
    key = keys_in[at];
    if (wave == 0) val = idx_in[at];
    // every 2^x-th sample: 64 per run (fewer of a run below 2^kMsTileLog)
    const int x = max(run_log - kMsTileLog, 0);
    const uint32_t have = n >> kSampleLog;
    uint32_t smp[kPer], len[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t b = (s0 + j) << run_log;
      len[j] = s0 + j == run || b >= n ? 0u : min(1u << run_log, n - b);
      const uint32_t s = (b >> kSampleLog) + ((lane + 1) << x) - 1;
      smp[j] = smp_in[s < have ? s : 0u];  // those past the run do not count
    }
    const uint32_t kf = lane_value(key, 0), kl = lane_value(key, 63);
    uint32_t lo[kPer], m[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const bool le = s0 + j < run;
      const uint32_t nc = len[j] >> (kSampleLog + x);
      lo[j] = count_below<kFull>(smp[j], kf, le, nc) << x;
      m[j] = count_below<kFull>(smp[j], kl, le, nc) << x;
    }
    uint32_t v[kPer], v2[kPer], v3[kPer];
    if (x > 0) {  // among the 2^x - 1 samples that follow
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const uint32_t b = ((s0 + j) << run_log) >> kSampleLog;
        const uint32_t s = b + lo[j] + lane, t = b + m[j] + lane;
        v[j] = smp_in[s < have ? s : 0u];
        v2[j] = smp_in[t < have ? t : 0u];
      }
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const bool le = s0 + j < run;
        const uint32_t ns = len[j] >> kSampleLog, most = (1u << x) - 1;
        lo[j] += count_below<kFull>(v[j], kf, le, min(ns - lo[j], most));
        m[j] += count_below<kFull>(v2[j], kl, le, min(ns - m[j], most));
      }
    }
    // the windows: m keys from w on
    const uint32_t *w[kPer];
    uint32_t wide = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      lo[j] <<= kSampleLog;
      m[j] = min((m[j] << kSampleLog) + kSample - 1, len[j]) - lo[j];
      w[j] = keys_in + (m[j] ? ((s0 + j) << run_log) + lo[j] : 0u);
      rank += lo[j];
      wide |= m[j] >= (uint32_t)kWindow ? 1u << j : 0u;
    }
    // to LDS, a window's last key repeated up to kWindow
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t top = max(m[j], 1u) - 1;
      v[j] = w[j][min(lane, top)];
      v2[j] = w[j][min(lane + 64, top)];
      v3[j] = w[j][min(lane + 128, top)];
    }
    uint32_t *win = s_win[wave];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      win[j * kWindow + lane] = v[j];
      win[j * kWindow + 64 + lane] = v2[j];
      win[j * kWindow + 128 + lane] = v3[j];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t pos[kPer];  // byte offset of the lower bound so far
#pragma unroll
    for (int j = 0; j < kPer; ++j) pos[j] = 0;
#pragma unroll
    for (int h = 1 << (kSteps - 1); h > 0; h >>= 1)
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const uint32_t y = *reinterpret_cast<const uint32_t *>(
            reinterpret_cast<const char *>(win) + pos[j] +
            4 * (j * kWindow + h - 1));
        pos[j] += sorts_below<kFull>(y, key, s0 + j < run) ? 4 * h : 0;
      }
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      rank += wide >> j & 1 ? 0u : min(pos[j] >> 2, m[j]);
    if (wide) {
      // each lane on its own, those runs side by side: its place among the
      // samples read above (in LDS), those between two, the keys that follow
      __builtin_amdgcn_wave_barrier();
      uint32_t p[kPer];
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        win[j * kWindow + lane] = smp[j];
        p[j] = 0;
        m[j] = wide >> j & 1 ? len[j] >> (kSampleLog + x) : 0u;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int step = 0; step < 7; ++step) {
#pragma unroll
        for (int j = 0; j < kPer; ++j)
          v[j] = win[j * kWindow + p[j] + (max(m[j] + 1, 2u) >> 1) - 1];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          p[j] += sorts_below<kFull>(v[j], key, s0 + j < run) ? (m[j] + 1) >> 1 : 0u;
          m[j] >>= 1;
        }
      }
      if (x > 0) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          p[j] <<= x;
          v2[j] = wide >> j & 1 ? min((1u << x) - 1, (len[j] >> kSampleLog) - p[j]) : 0u;
        }
        for (int step = 0; step < x; ++step) {
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            const uint32_t b = ((s0 + j) << run_log) >> kSampleLog;
            v[j] = smp_in[v2[j] ? b + p[j] + ((v2[j] + 1) >> 1) - 1 : 0u];
          }
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            p[j] += sorts_below<kFull>(v[j], key, s0 + j < run) ? (v2[j] + 1) >> 1 : 0u;
            v2[j] >>= 1;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        p[j] <<= kSampleLog;
        v2[j] = wide >> j & 1 ? min(kSample - 1, len[j] - p[j]) : 0u;
      }
      for (int step = 0; step < kSampleLog; ++step) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          const uint32_t b = (s0 + j) << run_log;
          v[j] = keys_in[v2[j] ? b + p[j] + ((v2[j] + 1) >> 1) - 1 : 0u];
        }
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          p[j] += sorts_below<kFull>(v[j], key, s0 + j < run) ? (v2[j] + 1) >> 1 : 0u;
          v2[j] >>= 1;
        }
      }
#pragma unroll
      for (int j = 0; j < kPer; ++j) rank += wide >> j & 1 ? p[j] - lo[j] : 0u;
    }
  }
  s_rank[wave][lane] = rank;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int g = 1; g < kWaves; ++g) rank += s_rank[g][lane];
  if (i < n) {
    const uint32_t to = (g0 << run_log) + (i - (run << run_log)) + rank;
    if (to < n) {  // always, with sorted runs
      keys_out[to] = key;
      idx_out[to] = val;
      if ((to & (kSample - 1)) == kSample - 1) smp_out[to >> kSampleLog] = key;
    }
  }
}

// Keys per tile, 2^this.  A block's rounds take 10-11 us at 2,048 keys, 16
// waves on one CU, and less with fewer on more CUs, while the merge of all the
// tiles stays one round.  Builds in us by tile of 2,048 / 1,024 / 512 keys:
// 2,500 triangles 26.3 / 23.4 / 22.1, 8,192 (caller bounds) - / 20.4 / 19.7,
// 16,384 31.1 / 28.3 / 28.8, 20,000 32.7 / 31.2 (heightfields 32.6 / 32.1), 32,768
// 33.1 / 31.4 (33.6 / 33.4); 64 tiles of 1,024 in one round turn, 65,536 37.2 /
// 38.3 (39.8 / 45.5).  One tile needs no merge: 1,024 triangles with caller bounds
// 16.2 / 15.4 / 17.7.
static int tile_log(const MergeKeys &src, uint32_t n) {
  if (n <= 1u << 10) return n <= 1u << 9 ? 9 : 10;
  if (src.whole) return kMsTileLog;
  return n <= 16u << 9 ? 9 : n <= 32u << 10 ? 10 : kMsTileLog;
}

// The merge rounds of a sort of n keys: up to 32 tiles merge in one round, eight
// waves per 64 keys, since their searches in a row are its time (builds of
// 50,000 39.4 us with four waves, 37.7 with eight; heightfields 40.3, 38.1).
// More tiles merge 16 runs at a time, four waves (with one, for 8 runs, 66,000
// triangles took 46.6 us, with four 42.0), before a last round of up to 16; with
// eight waves 2^18 triangles take 66.5 us, not 63.4.
struct MergeRound {
  int run_log;          // runs of 2^run_log keys
  int group_log;        // 2^group_log of them merged together
};
constexpr int kMaxMergeRounds = 8;
static int merge_plan(const MergeKeys &src, uint32_t n, MergeRound *r) {
  int rounds = 0, log = tile_log(src, n);
  uint32_t runs = (n + (1u << log) - 1) >> log;
  while (runs > 1) {
    int g = 4;
    if (runs <= (rounds ? 16u : 32u))
      for (g = 3; 1u << g < runs;) ++g;
    r[rounds++] = {log, g};
    runs = (runs + (1u << g) - 1) >> g;
    log += g;
  }
  return rounds;
}

// Sample words of one buffer; a sort's samples are two.
static uint32_t merge_samples(uint32_t n) { return (n >> kSampleLog) + 1; }
static_assert(kMergeBuildMax <= 16u << kMaxRunLog, "the last round's runs");
static_assert(2 * ((kSmallSortTile >> kSampleLog) + 1) <= 2 * kRadix,
              "a radix sort's count words per tile hold its samples");

void launch_tile_sort(const MergeKeys &src, uint32_t n, uint32_t *keys_tmp,
                      int32_t *idx_tmp, uint32_t *keys_out, int32_t *idx_out,
                      uint32_t *samples, hipStream_t s) {
  // the tile sort and every round alternate buffers, the last one writes out
  MergeRound rounds[kMaxMergeRounds];
  const bool odd = merge_plan(src, n, rounds) % 2;
  uint32_t *k = odd ? keys_tmp : keys_out;
  int32_t *v = odd ? idx_tmp : idx_out;
  const int log = tile_log(src, n);
#define LBVH_TILE_SORT(SRC, FULL, T)                                      \
  hipLaunchKernelGGL((k_tile_sort<SRC, FULL, T>), dim3((n + T - 1) / T),  \
                     dim3(T / kMsPer), 0, s, src, n, k, v, samples)
#define LBVH_TILE_SORTS(SRC, FULL)                       \
  do {                                                   \
    if (log == 9) LBVH_TILE_SORT(SRC, FULL, 512);        \
    else if (log == 10) LBVH_TILE_SORT(SRC, FULL, 1024); \
    else LBVH_TILE_SORT(SRC, FULL, kMsTile);             \
  } while (0)
  if (src.keys) LBVH_TILE_SORTS(kSrcKeys, true);
  else if (src.cen) LBVH_TILE_SORTS(kSrcCentres, false);
  else if (src.whole) LBVH_TILE_SORTS(kSrcWholeMesh, false);
  else LBVH_TILE_SORTS(kSrcTriangles, false);
#undef LBVH_TILE_SORTS
#undef LBVH_TILE_SORT
}

template <bool kFull>
static void merge_rounds(const MergeKeys &src, uint32_t n, uint32_t *keys_tmp,
                         int32_t *idx_tmp, uint32_t *keys_out, int32_t *idx_out,
                         uint32_t *samples, hipStream_t s) {
  MergeRound rounds[kMaxMergeRounds];
  const int count = merge_plan(src, n, rounds);
  const bool odd = count % 2;
  uint32_t *smp = samples, *smp2 = samples + merge_samples(n);
  uint32_t *k = odd ? keys_tmp : keys_out, *k2 = odd ? keys_out : keys_tmp;
  int32_t *v = odd ? idx_tmp : idx_out, *v2 = odd ? idx_out : idx_tmp;
  for (int r = 0; r < count; ++r) {
    const int run_log = rounds[r].run_log, g = rounds[r].group_log;
#define LBVH_MERGE(WAVES, PER)                                            \
  hipLaunchKernelGGL((k_merge<WAVES, PER, kFull>), dim3((n + 63) / 64),   \
                     dim3(64 * WAVES), 0, s, k, v, smp, k2, v2, smp2, n, \
                     run_log)
    if (count == 1) {
      if (g == 5) LBVH_MERGE(8, 4);
      else if (g == 4) LBVH_MERGE(8, 2);
      else LBVH_MERGE(8, 1);
    } else {
      if (g == 4) LBVH_MERGE(4, 4);
      else LBVH_MERGE(4, 2);
    }
#undef LBVH_MERGE
    std::swap(k, k2);
    std::swap(v, v2);
    std::swap(smp, smp2);
  }
}

void launch_merge_rounds(const MergeKeys &src, uint32_t n, uint32_t *keys_tmp,
                         int32_t *idx_tmp, uint32_t *keys_out,
                         int32_t *idx_out, uint32_t *samples, hipStream_t s) {
  if (src.keys)
    merge_rounds<true>(src, n, keys_tmp, idx_tmp, keys_out, idx_out, samples, s);
  else
    merge_rounds<false>(src, n, keys_tmp, idx_tmp, keys_out, idx_out, samples, s);
}

}  // namespace lbvh
