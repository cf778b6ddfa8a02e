// spl_internal.h -- host-side declarations shared by the C-ABI layer and the
// kernel translation units.
//
// Every stage runs for a batch of views at once: per-view buffers live in
// one allocation each, view v at base + v * stride, and kernels take the view
// from blockIdx.y (or loop over views where one read of the scene serves all
// of them: cull and project).  A single frame is the batch of one.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace spl {

// Frame uniforms: renderer.rs:49-61 plus the frame's tile grid.
struct Uniforms {
  float camera_matrix[16];
  float view_matrix[16];
  float view_projection_matrix[16];
  float view_size[2];
  uint32_t image_size[2];
  float frustum_culling_tolerance;
  float ellipse_size_bias;
  float ellipse_margin;
  float splat_scale;
  uint32_t tiles_x, tiles_y;
};

constexpr int kTileSize = 16;        // raster tile edge in pixels (16x16 = 256 lanes)
// Neighbouring screen tiles that the raster gives to one XCD before the next
// XCD's run.  Short, because views are uneven: with an eighth of the screen to
// each XCD, the one with the horizon was still at work when the ones with the
// sky were done (16 views of 6M splats: a pass of 12.84 ms so, 11.50 with
// runs of 4, 11.65 with 16, 11.48 with 120; one 4K view 1.57, 1.48, 1.45 and
// 1.47 ms; one 1080p view of 1M 561, 550, 562 and 565 us).
constexpr uint32_t kXcdRun = 4;
constexpr int kMaxDepthPasses = 4;   // 30-bit depth keys: 4 x 8 bits or 3 x 10 bits
constexpr int kMaxPairPasses = 3;    // screen-tile ids up to 24 bits
constexpr int kRecordFloat4 = 3;     // 48-byte record: rgba | A00 A10 A01 A11 | tx ty box box
constexpr int kMaxViews = 32;        // views per launch (one bit each in the visibility masks)

// Counter block layout (u32 words), one block per view.
enum CounterSlot : int {
  kCtrCull = 0,     // view 0's block holds the shared multi-view cull counters
  kCtrSort0 = 1,    // .. kCtrSort0 + 3
  kCtrBin = 5,
  kCtrPair0 = 6,    // .. kCtrPair0 + 2
  kCtrCount = 9,
  kVisible = 32,
  kPairs = 33,
  kPairOverflow = 34,
  kScatterError = 35,
  kHeavyAll = 36,   // view 0's block: tiles that k_heavy_tiles found heavy
  kHeavyTiles = 37, // .. + kHeavyClasses - 1: tiles in each of its lists
  kLongTiles = 41,  // view 0's block: tiles that start first among the ordinary ones
  kCounterWords = 64
};

// Heavy tiles: lists of at least kHeavyMin pairs and 1 / kHeavyShare of the
// batch's pairs, rounded down, so kHeavyCap of them but for rounding (1001 lists
// of 512 pairs): one past the cap stays an ordinary tile.  An ordinary block
// takes about 11 ns for each entry of its list, the device about 25 entries a
// ns over all tiles: a list of 1/275 of the pairs lasts as long as the whole
// raster.  The share is some four times that, because a frame saturates most
// tiles early and the long lists cluster on screen; us a pass at 1/400, 1/900,
// 1/1400 and 1/2500: 6M splats at 1080p 1180, 1127, 1090, 1549; 1M 540, 530,
// 525, 598; 1.5M at VGA 462, 455, 467, 465; five views of 300k 575, 535, 537,
// 665 (at 1/2500 they are too many for the eightfold reading to pay).
constexpr uint32_t kHeavyShare = 1000, kHeavyMin = 512, kHeavyCap = 1000;
// Of the others, those of a quarter of that and twice the view's mean list
// start first (kLongCap of them at most).
constexpr uint32_t kLongCap = 2048;
constexpr int kHeavyClasses = 4;
constexpr uint32_t kHeavyFlag = 0x80000000u;  // in a tile range's start (starts are below 2^30)

// Scene data in HBM, one stream per attribute (structure of arrays).
struct SceneView {
  const float* centers;     // 3 floats per splat, packed
  const float4* rotations;  // (r, i, j, k) normalised
  const float4* scale_alpha;// exp-scale xyz, sigmoid alpha
  const float* sh;          // 48 floats per splat, coefficient-major RGB
  uint32_t count;
};

// shaders.wgsl:249-266: the spherical-harmonics basis constants.  A scene
// stores coefficient k of every colour channel multiplied by constant k
// (the product each term of the reference's lookup starts with).
constexpr float kShConstants[16] = {
    0.28209479177387814f, -0.4886025119029199f, 0.4886025119029199f, -0.4886025119029199f,
    1.0925484305920792f, -1.0925484305920792f, 0.31539156525252005f, -1.0925484305920792f,
    0.5462742152960396f, -0.5900435899266435f, 2.890611442640554f, -0.4570457994644658f,
    0.3731763325901154f, -0.4570457994644658f, 1.445305721320277f, -0.5900435899266435f,
};

constexpr int kCullThreads = 256, kCullItems = 16;   // 4096 splats per cull / project tile
constexpr int kSortTile = 4096;                      // keys per sort tile: 4096, 8192 or 16384,
constexpr int kSortTileSmall = 1024;                 // or these, for one view of a small scene:
constexpr uint32_t kSmallSort = 7u << 14;            // its splats (depth sort, 8-bit digits)
constexpr uint32_t kSmallPairs = 1u << 15;           // and (pair sort, with a capacity
constexpr uint32_t kSmallPairCap = 1u << 20;         // of no more pairs than this)
constexpr int kTileNarrow = 8192, kTileWide = 16384; // by_count_tile's two,
constexpr int kTileByCount = 1;                      // asked for by this tile size
constexpr int kBinThreads = 256, kBinItems = 4;      // 1024 draw ranks per bin tile, 256 in small batches
constexpr uint32_t kHistCopies = 8;                  // of each view's digit histograms, summed by the sort
constexpr int kCullTile = kCullThreads * kCullItems;

struct CullLaunch {
  const float* centers;
  uint32_t n;
  uint32_t views;
  const Uniforms* uniforms;  // [views]
  int gpu_predicate;         // 1: shaders.wgsl:54-61 (DepthSorting::None), 0: renderer.rs:381-387
  int write_keys;
  uint32_t* keys; size_t keys_stride;        // view v: keys + v * keys_stride
  uint32_t* idx; size_t idx_stride;
  uint32_t* vis;                             // [n] visibility mask over views
  uint32_t* tile_prefix; size_t tp_stride;   // [views][cull tiles] exclusive prefix
  uint32_t* status; size_t status_stride;    // [views][cull tiles]
  uint32_t* counters;                        // [views][kCounterWords]
  uint32_t* hist;                            // one view: kHistCopies digit histograms; null: not here
  size_t hist_copy;                          // words between them
  int bits;
  int grid;
};

struct HistLaunch {
  const uint32_t* keys; size_t keys_stride;
  uint32_t* hist; size_t hist_stride;        // [views][passes << bits]
  uint32_t* counters;
  int passes, bits;
  uint32_t* clear; size_t clear_words; size_t clear_stride;  // per view
  int grid_x, views;
};

struct SortPassLaunch {
  const uint32_t* keys_in;
  const uint32_t* vals_in;   // null: values are the input positions
  uint32_t* keys_out;
  uint32_t* vals_out;
  size_t entry_stride;       // per view, all four arrays
  uint32_t* counters;        // [views][kCounterWords]
  int count_slot;            // kVisible or kPairs
  uint32_t count_cap;
  int shift;
  const uint32_t* hist; size_t hist_stride;  // this pass's histogram, per view
  size_t hist_copy;          // words between its kHistCopies copies
  uint32_t* status; size_t status_stride;    // [tiles][radix], per view
  int tile_slot;             // counter slot of this pass's tile counter
  uint32_t* clear_a; size_t clear_a_words; size_t clear_a_stride;
  uint32_t* clear_b; size_t clear_b_words; size_t clear_b_stride;
  uint32_t clear_a_tile;     // keys per tile of the status at clear_a (used_status); 0: clear_a_words it is
  uint32_t one_round;        // keys of one round of 1024-lane blocks, one a CU, in tiles of kTileNarrow
  int tile_keys;             // 1024, 4096, 8192, 16384 or kTileByCount
  int few;                   // few keys in all: more lanes with fewer keys each
  int grid_x, views;
};

struct ProjectLaunch {
  SceneView scene;
  uint32_t views;
  const Uniforms* uniforms;
  const uint32_t* vis;
  const uint32_t* tile_prefix; size_t tp_stride;
  uint32_t parts;                           // blocks that share a cull tile: 1, 2, 4, 8 or 16
  int sh_order;
  int use_covariance_for_scale;
  int use_unaligned_rectangles;
  float4* records; size_t rec_stride;       // float4 units per view
  uint2* boxes; size_t box_stride;          // pixel box per entry, dense, for the binning
  double* conics;                           // optional, view 0 only, 6 per entry
  uint32_t* clear_a; size_t clear_a_words; size_t clear_a_stride;
  uint32_t* clear_b; size_t clear_b_words; size_t clear_b_stride;
  int grid;
};

struct BinLaunch {
  const uint32_t* order; size_t order_stride;  // record index per draw rank; null = identity
  const uint2* boxes; size_t box_stride;       // pixel box per record
  const Uniforms* uniforms;
  uint32_t* pair_keys;
  uint32_t* pair_vals; size_t pair_stride;
  uint32_t pair_cap;
  uint32_t* hist; size_t hist_stride;          // [kHistCopies][kMaxPairPasses][256] per view, accumulated
  int pair_passes;
  uint64_t* status; size_t status_stride;
  uint32_t* counters;
  // finished bookkeeping of the depth sort, zeroed here (per view)
  uint32_t* clear_a; size_t clear_a_words, clear_a_stride;
  uint32_t* clear_b; size_t clear_b_words, clear_b_stride;
  int items;                                   // entries a lane: kBinItems or 1
  int grid_x, views;
};

struct RangesLaunch {
  const uint32_t* pair_keys; size_t pair_stride;
  uint32_t* counters;
  uint32_t pair_cap;
  const Uniforms* uniforms;
  uint2* ranges; size_t ranges_stride;
  uint32_t* clear_a; size_t clear_a_words; size_t clear_a_stride;
  uint32_t clear_a_tile, one_round;  // as in SortPassLaunch
  uint32_t* clear_b; size_t clear_b_words; size_t clear_b_stride;
  int grid_x, views;
};

struct HeavyLaunch {
  uint2* ranges; size_t ranges_stride;
  const Uniforms* uniforms;
  uint32_t* counters;
  uint32_t pair_cap;
  uint32_t* list;                            // kHeavyClasses lists of kHeavyCap, one of kLongCap: view << 24 | tile
  uint32_t long_cap;                         // most of those listed: kLongCap, or all tiles
  uint32_t heavy_cap;                        // most tiles listed: kHeavyCap, or all tiles
  uint2* tile_work;                          // optional, view 0, as in RasterLaunch
  uint32_t max_tiles;
  int views;
};

struct RasterLaunch {
  const uint32_t* heavy;     // k_heavy_tiles' lists
  uint32_t heavy_cap, long_cap;
  uint32_t slots_per_view;   // multiple of 8 * kXcdRun, >= the largest view's tile count
  const uint32_t* pair_vals; size_t pair_stride;
  const float4* records; size_t rec_stride;
  uint2* ranges; size_t ranges_stride;
  const Uniforms* uniforms;
  uint32_t* const* pixels;   // [views] frame buffers
  uint32_t* counters;
  int use_unaligned_rectangles;
  int blend_f32;
  int walk;                  // raster mode: 0 entry-major per quadrant, 1 per-pixel walk, 2 per 4x4 sub-block,
                             // 3 per-lane walk over coverage masks
  int batch_entries;         // entries staged in LDS per batch: 128 or 256
  int bgra;
  uint2* tile_work;          // optional, view 0: per tile (list length, entries consumed)
  int grid_x, views;
};

void launch_cull(const CullLaunch& a, hipStream_t s);
void launch_histograms(const HistLaunch& a, hipStream_t s);
void launch_sort_pass(int bits, const SortPassLaunch& a, hipStream_t s);
void launch_project(const ProjectLaunch& a, hipStream_t s);
void launch_bin(const BinLaunch& a, hipStream_t s);
void launch_ranges(const RangesLaunch& a, hipStream_t s);
void launch_heavy_tiles(const HeavyLaunch& a, hipStream_t s);
void launch_raster(const RasterLaunch& a, hipStream_t s);

// Writes a batch's uniforms and frame pointers with one kernel that carries
// them in its arguments; false for more views than those hold.
bool launch_upload(const Uniforms* u, uint32_t* const* pixels, uint32_t views, Uniforms* d_uniforms,
                   uint32_t** d_pixels, hipStream_t s);

// spl_render_frame_static: the scratch array's size and the largest scene and
// frame it takes.
constexpr uint64_t kStaticScratchBytes = 52ull << 20;
constexpr uint32_t kStaticMaxSplats = 1u << 17;
constexpr uint32_t kStaticMaxWidth = 3840, kStaticMaxHeight = 2160;
// Writes the frame's uniforms and pixel pointer and zeroes `zero_words`
// words at `zero` (the bookkeeping that starts every frame at zero), with
// one kernel.
void launch_static_setup(const Uniforms& u, uint32_t* pixels, Uniforms* d_uniforms, uint32_t** d_pixels,
                         uint32_t* zero, size_t zero_words, hipStream_t s);

}  // namespace spl
