// lbvh_internal.h -- shared definitions of the HIP kernels and the host API.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lbvh {

// ---- sizes and launch shapes --------------------------------------------

// Sort digits: 8 bits (4 passes over the 30-bit Morton keys: bits 0-7,
// 8-15, 16-23, 24-29) or, as a tunable, 10 bits (3 passes: 0-9, 10-19,
// 20-29).  The stand-alone sort takes any u32 key: 4 passes of 8 bits, or of
// 10 bits (the last one 2 bits wide) when that width is fixed.
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;  // 256 digit values per pass
constexpr int kWideBits = 10;
constexpr int kWideRadix = 1 << kWideBits;
constexpr int kKeyBits = 30;      // Morton keys
constexpr int kFullKeyBits = 32;  // keys of the stand-alone sort
constexpr int kHistWords = 4 * kWideRadix;  // >= passes x digits of any sort
__host__ __device__ constexpr int sort_passes(int bits,
                                             int key_bits = kKeyBits) {
  return (key_bits + bits - 1) / bits;
}
__host__ __device__ constexpr int sort_radix(int bits) { return 1 << bits; }
static_assert(sort_passes(kRadixBits) * kRadix <= kHistWords, "hist size");
static_assert(sort_passes(kWideBits) * kWideRadix <= kHistWords, "hist size");
static_assert(sort_passes(kRadixBits, kFullKeyBits) * kRadix <= kHistWords,
              "hist size");
static_assert(sort_passes(kWideBits, kFullKeyBits) * kWideRadix <= kHistWords,
              "hist size");
constexpr int kSortThreads = 256;        // 4 wave64 per tile
constexpr int kSortItems = 16;           // keys per thread
constexpr int kSortTile = kSortThreads * kSortItems;  // 4096 keys per tile
// A single-mesh sort of at most kSmallSortMax keys uses tiles of
// kSmallSortTile keys (4 per thread): a small sort is a chain of one-tile
// latencies, and a quarter of the serial work per thread shortens each
// (builds of 2^16 / 2^17 / 2^18 triangles 0.092 / 0.105 / 0.115 -> 0.076 /
// 0.087 / 0.100 ms); above 2^20 keys the four times longer count columns
// cost more than the shorter tiles save.
constexpr int kSmallSortItems = 4;
constexpr int kSmallSortTile = kSortThreads * kSmallSortItems;  // 1024 keys
constexpr uint32_t kSmallSortMax = 1u << 20;
// Batched sorts of at most this many keys in all use the small tile too: 17,555
// keys in 16 meshes 81.6 / 61.9 us a batch, 713,000 in 300 141 / 107, 4.8M in
// 700 450 / 429 (4,096 / 1,024 keys); 18M in 1,000 turns, 1,438 / 1,535.
// But one block scans a mesh's tile counts, so a large mesh's small tiles are a
// long chain, with 10-bit digits, whose tiles hold four times the counts, the
// longer, and less so in four groups of threads (seg_scan_groups): the meshes must
// have at most so many keys each.  Batches in us, 4,096 / 1,024 keys.
//   8 bits, up to kSmallSortMax in all: 65,536 with 200 meshes of 2,000 125 / 122,
//   131,072 with those 144 / 164; in four groups 200,000 alone 132 / 116, 5 of them 171 /
//   170, 131,072 with 40 of 2,000 130 / 102, 4 of 262,144 163 / 181.  More in all: 100 of
//   32,768 290 / 285, 60 of 65,536 329 / 340, 5M alone 634 / 1,226.
//   10 bits: 16,384 with 300 of 300 89 / 83, 24,576 with those 96 / 96; in four groups
//   20,000 alone 96 / 84, 32,768 alone 91 / 101, 100,003 alone 128 / 187.  More in all: 280
//   of 4,096 144 / 133, 500 of 4,096 187 / 190, 240 of 8,192 187 / 201, 1M with 500 of
//   2,000 530 / 1,433.
constexpr uint32_t kBatchSmallMax = 1u << 23;
inline uint32_t batch_small_mesh(uint32_t n, int bits, int groups) {
  if (n > kSmallSortMax) return bits == kWideBits ? 1u << 12 : 1u << 15;
  if (groups == 1) return bits == kWideBits ? 1u << 14 : 1u << 16;
  return bits == kWideBits ? 5u << 12 : 3u << 16;
}
// Groups of threads that share a mesh's scan (k_seg_scan).  One takes 9 us for a
// mesh of 64 tiles, the chain of its loads, four 5; but four where blocks fill the
// chip cost more (300 meshes 4.8 against 3.6 us, 1,000 8.8 against 6.2).
inline int seg_scan_groups(uint32_t num_segs, uint32_t tiles) {
  return num_segs <= 256 && tiles > 4 * num_segs ? 4 : 1;
}

constexpr int kTreeTileDefault = 1024;  // leaves per tile of the fused up pass
constexpr int kMaxTreeLevels = 16;      // agglomeration levels (6 at 2^24, T=1024)
constexpr int kTreeFrontier = 128;      // item slots per agglomeration tile
constexpr int kItemInt4 = 3;            // 48-byte items: range, box, gap deltas

constexpr int kMapThreads = 256;  // triangle-parallel kernels
// Grid of the bounds reduction, two blocks per CU.  So few partials are
// folded by the kernel that makes the keys, each block for itself, which saves
// builds a launch and the one-block fold's latency (2-5 us: 2^18 triangles
// 71.3 -> 69.4 us, 2^20 155.8 -> 153.3, 2^22 387 -> 382); more blocks stream no
// faster (2^24 1,319 -> 1,318 us against 2,048).
constexpr int kBoundsBlocks = 512;
constexpr int kMortonBlocksMax = 2048;  // grid-stride Morton (per-stage entry)

// ---- device control block ------------------------------------------------
//
// One per context, zeroed at allocation.  Nothing in it needs a reset
// between operations (or graph replays):
//   fault       sticky bits (kFault*), never set in a correct run; read and
//               cleared by lbvh_synchronize
//   bounds      scene bounds of the last stand-alone reduction
//   hist        global digit counts of each pass of the current sort (pass
//               p's at hist + p * radix)
constexpr uint32_t kFaultUpFrontier = 4u;  // per-stage up pass: a block left
                                           // more than kUpFront items, or
                                           // the last level left items
constexpr uint32_t kFaultFrontier = 8u;    // agglomeration frontier overflow
constexpr uint32_t kFaultNotATree = 16u;   // per-stage up pass: an index or
                                           // parent out of range, a path
                                           // longer than any tree's, a third
                                           // child at a node, or a root that
                                           // never merged
struct Ctl {
  uint32_t fault;
  uint32_t pad0[7];
  float bounds[8];                       // min.xyz, 0, max.xyz, 0
  uint32_t hist[kHistWords];             // global digit counts per pass
};


// Morton quantisation parameters (uniform block of aabb-z-idx.js:164-169).
struct MortonParams {
  float bmin[3];
  float ext[3];  // max - min
  float rcp[3];  // fl(1 / ext)
  int div_mode;  // lbvh_div_mode
};

// ---- kernel launchers (each .hip file owns its kernels) --------------------

// k_bounds_morton.hip
// Scene bounds into ctl->bounds; cen (3 x cen_stride(n) floats, or null):
// also each triangle's box centre, and the partials are left to the kernel
// that reads the centres.  Returns their number.
uint32_t launch_bounds(const float4 *tri, uint32_t n, float4 *partials,
                       Ctl *ctl, hipStream_t s, float *cen = nullptr);
// Morton keys + per-tile digit counts (as launch_aabb_morton with cnt) from
// the centres launch_bounds wrote and its `parts` partials.
void launch_morton_cen(const float *cen, uint32_t n, int div_mode,
                       uint32_t *keys, uint32_t *cnt, int bits, hipStream_t s,
                       const float4 *partials, uint32_t parts);
// Box centres: x, y and z arrays of cen_stride(n) floats each (a multiple of
// 64, so every array and every 256-triangle chunk starts 256-byte aligned
// and is read and written 16 bytes per lane).
__host__ __device__ constexpr uint32_t cen_stride(uint32_t n) {
  return (n + 63u) & ~63u;
}
// cnt (sort_radix(bits) x sort_tiles(n) words, or null): also write the
// first sort pass's per-tile digit counts for digits of `bits` bits.
void launch_aabb_morton(const float4 *tri, uint32_t n, const MortonParams &p,
                        bool bounds_from_ctl, float4 *aabb, uint32_t *keys,
                        Ctl *ctl, hipStream_t s, uint32_t *cnt = nullptr, int bits = kRadixBits);
void launch_copy_bounds(const Ctl *ctl, float *out, hipStream_t s);

// k_sort.hip
// Segments of a batched sort (all null: one segment [0, n)).  Tiles of
// kSortThreads x items keys never straddle segments; tile_seg maps each tile to its
// segment, seg_tile0 gives a segment's first tile, seg_off its first key
// (S+1 entries).
struct SortSegs {
  const uint32_t *tile_seg;
  const uint32_t *seg_tile0;
  const uint32_t *seg_off;
  int items;  // keys per thread of the tiles
};
// One digit pass of `bits`-bit digits (kRadixBits or kWideBits) over
// `tiles` sort tiles (pass 0 takes the position in the segment as payload
// and ignores vals_in).  cnt and off hold sort_radix(bits) x tiles words
// each; counted: cnt already holds this pass's per-tile digit counts (the
// Morton kernels write pass 0's).  A single mesh takes its digit bases from
// the column sums of cnt (into ctl->hist); each segment from its own tiles'
// counts, in one block per segment.  keys_in and keys_out must differ.
// key_bits: significant bits of the keys (a digit with few of them is
// counted with matched lanes).
void launch_sort_pass(int bits, int pass, const uint32_t *keys_in,
                      const int32_t *vals_in, uint32_t *keys_out,
                      int32_t *vals_out, uint32_t n, uint32_t tiles,
                      uint32_t *cnt, uint32_t *off, bool counted, Ctl *ctl,
                      hipStream_t s, const SortSegs *segs = nullptr,
                      uint32_t num_segs = 0, int key_bits = kKeyBits);
// Keys per thread and tiles of a single-mesh sort of n keys.
inline int sort_items(uint32_t n) {
  return n <= kSmallSortMax ? kSmallSortItems : kSortItems;
}
inline uint32_t sort_tiles(uint32_t n) {
  const uint32_t t = (uint32_t)(kSortThreads * sort_items(n));
  return (n + t - 1) / t;
}
// Tiles of one mesh of a batched sort.
inline uint32_t batch_sort_tiles(uint32_t n, int items) {
  const uint32_t t = (uint32_t)(kSortThreads * items);
  return (n + t - 1) / t;
}
// The sort of a single key: perm[0] = 0 and sorted[0] = keys[0] (sorted may
// be keys).  A one-thread kernel, so that a build stays kernels only.
void launch_single_key(const uint32_t *keys, uint32_t *sorted, int32_t *perm,
                       hipStream_t s);

// k_merge_sort.hip
// A sort of at most kMergeSortMax keys, or a build's of at most kMergeBuildMax,
// goes by tiles of up to kMsTile keys in LDS and rank merges of the tiles, not
// by radix passes: one merge round up to 32 tiles, two beyond.  A build saves
// its Morton launch too, so its line lies higher.  Builds of uniform meshes in
// us, merged / by the better digit width: 66,000 41.8 / 60.9, 2^17 48.1 / 65.5,
// 2^18 63.7 / 79.8, 300,000 75.5 / 87.0, 393,216 87.2 / 96.2 (heightfields 43.6 /
// 60.3, 50.3 / 63.7, 63.3 / 75.3, 77.7 / 85.9, 90.1 / 93.0), 2^19 107.9 / 104.9;
// sorts of random keys 66,000 23.0 / 45.5, 2^18 35.7 / 46.3, 280,000 49.1 / 47.6.
constexpr int kMsTileLog = 11;
constexpr int kMsTile = 1 << kMsTileLog;
constexpr uint32_t kMergeSortMax = 128u << kMsTileLog;
constexpr uint32_t kMergeBuildMax = 192u << kMsTileLog;
// The keys of a merge sort: given (any u32; `keys` may be the output), or
// Morton keys made by the tile sort -- from the centres launch_bounds wrote
// with the bounds folded from its `parts` partials, from the triangles with the bounds in p, or (whole: n <= kMsTile) from the triangles
// with the bounds of the one tile.
struct MergeKeys {
  const uint32_t *keys;
  const float *cen;
  const float4 *tri;
  const float4 *partials;
  uint32_t parts;
  int whole;
  MortonParams p;
};
// The tile sort, then the merge rounds, both given the same buffers: the
// sorted keys and their input positions end in keys_out and idx_out.
// samples: n / 16 + 2 words (a sort's digit counts and offsets are more).
void launch_tile_sort(const MergeKeys &src, uint32_t n, uint32_t *keys_tmp,
                      int32_t *idx_tmp, uint32_t *keys_out, int32_t *idx_out,
                      uint32_t *samples, hipStream_t s);
void launch_merge_rounds(const MergeKeys &src, uint32_t n, uint32_t *keys_tmp,
                         int32_t *idx_tmp, uint32_t *keys_out,
                         int32_t *idx_out, uint32_t *samples, hipStream_t s);

// k_tree.hip
// The per-stage radix tree (parents array) in three launches over 4,096-gap
// tiles; scratch of radix_tree_scratch_bytes(n) (spine records, per-tile
// summaries), nothing in it needs clearing.
uint64_t radix_tree_scratch_bytes(uint32_t n);
void launch_radix_tree(const uint32_t *keys, uint32_t n, int32_t *parents,
                       void *scratch, hipStream_t s);
// Per-stage up pass: the level-1 kernel, then item levels until one block
// holds the root; scratch of up_pass_scratch_bytes(n) (items, then counts).
uint64_t up_pass_scratch_bytes(uint32_t n);
void launch_up_pass(const int32_t *idx, const float4 *aabb,
                    const int32_t *parents, uint32_t n, float4 *nodes,
                    void *scratch, Ctl *ctl, hipStream_t s);
void launch_rearrange(const float4 *tri, const int32_t *idx, uint32_t n,
                      float4 *out, hipStream_t s);
// Segments of one agglomeration level of a batched build (all null: one
// mesh).  Per tile of the level: its segment; per segment: its first tile at
// this level, its first leaf (seg_off, S+1 entries), and (levels >= 1) its
// first tile and tile count at the level below.
struct TreeSegs {
  const uint32_t *tile_seg;
  const uint32_t *seg_tile0;
  const uint32_t *seg_off;
  const uint32_t *prev_tile0;
  const uint32_t *prev_tiles;
};

// Fused leaf gather + radix tree + node boxes by multi-level agglomeration:
// level 0 over tiles of `tile` (256, 512 or 1024) sorted leaves, then item
// levels until one tile remains.  Tiles are numbered level after level; the
// item slots hold kTreeFrontier items of kItemInt4 int4 per tile and the
// counts one word per tile (tree_tiles_total(n, tile) tiles).
//
// Tiles of each level of an n-leaf build (returns the number of levels).
int tree_levels(uint32_t n, int tile, uint32_t *grid);
uint64_t tree_tiles_total(uint32_t n, int tile);
// Level 0 by climbs (k_leaves), over leaf tiles of `tile` (batched builds pass
// their segments).
void launch_leaves(int tile, uint32_t grid, const float4 *tri,
                   const uint32_t *skeys, const int32_t *perm, uint32_t n,
                   float4 *otri, int4 *items_out, uint32_t *count_out,
                   float4 *nodes, Ctl *ctl, const TreeSegs &segs,
                   hipStream_t s);

// k_forest.hip
// Level 0 of at most kForestMax leaves in all, without climbs, over leaf tiles of
// kForestTile.  Refits in us, this / k_leaves' tile of 1,024 under the same item
// levels: 20,000 leaves 15.9 / 17.5, 2^16 16.4 / 21.9, 2^18 24.8 / 26.2, 500,000 40.4
// / 36.1 (the last of two rounds of tiles is short), 1M 61.2 / 58.7, 3M 145 / 144;
// heightfields 15.5 / 18.2, 16.7 / 23.3, 23.0 / 24.1, 33.9 / 31.1, 46.5 / 51.7, 98.5 /
// 107, which turn at 3.6M (3.9M 158 / 140).
constexpr int kForestTile = 256;
constexpr uint32_t kForestMax = 7u << 19;
void launch_forest_leaves(uint32_t grid, const float4 *tri,
                          const uint32_t *skeys, const int32_t *perm,
                          uint32_t n, float4 *otri, int4 *items_out,
                          uint32_t *count_out, float4 *nodes, Ctl *ctl,
                          const TreeSegs &segs, hipStream_t s);
// An item level, over either leaf level.  items_in / count_in: the level below's
// slots and counts, indexed by its tile number; prev_tiles: its tile count (one
// mesh).
void launch_items(uint32_t grid, uint32_t n, const int4 *items_in,
                  const uint32_t *count_in, uint32_t prev_tiles,
                  int4 *items_out, uint32_t *count_out, float4 *nodes, Ctl *ctl,
                  const TreeSegs &segs, hipStream_t s);

// k_batch.hip
// The blocks of a batch's bounds: each block's mesh, and each mesh's first block
// (S + 1 entries).  A mesh has one per sort tile, at most kBoundsBlocks.
struct BoundsBlocks {
  const uint32_t *blk_seg;
  const uint32_t *seg_blk0;
};
// Per-mesh bounds, two float4 each at the mesh's first block in `folded` (as
// large as partials: two float4 a block), and box centres (3 x total floats).
void launch_batch_bounds(const float4 *tri, const uint32_t *seg_off,
                         const BoundsBlocks &blocks, uint32_t grid,
                         uint32_t num_segs, float4 *partials, float4 *folded,
                         float *cen, uint32_t total, hipStream_t s);
// Per-mesh Morton keys and the first sort pass's per-tile digit counts;
// centres from cen when non-null, else from tri.
void launch_batch_morton(const float4 *tri, const float *cen, uint32_t total,
                         const SortSegs &segs, uint32_t tiles,
                         const float *seg_bounds, const BoundsBlocks &blocks,
                         const float4 *folded, int div_mode, uint32_t *keys,
                         uint32_t *cnt0, int bits, hipStream_t s);

// k_raycast.hip
void launch_raycast(const void *nodes, const float *tri, uint32_t n,
                    const float *rays, uint32_t count, float *hits,
                    hipStream_t s);

}  // namespace lbvh

// lbvh_api.hip: a context's device control block, for the server's
// per-request epilogue (which reads and clears its fault word).
struct lbvh_ctx;
lbvh::Ctl *lbvh_context_ctl(lbvh_ctx *ctx);
