// raster.hip -- compute rasteriser for the projected rectangles.
//
// Replaces the fixed-function half of the reference's render pass
// (renderer.rs:247-291,435-455) and its fragment stage (shaders.wgsl:580-592):
//  bin     one (screen tile, record) pair per 16x16 tile a splat's pixel box
//          touches, written in draw order (single-pass scan with decoupled
//          look-back, pairs emitted by a balanced block-wide expansion), plus
//          the digit histograms of the tile ids for the stable pair sort.
//  ranges  [start, end) of each tile's run in the tile-sorted pair list.
//  raster  one 256-lane block per tile, one lane per pixel, one wave per 8x8
//          quadrant: records staged in LDS 128 or 256 at a time, each wave
//          keeping the ones that can reach its still-transparent pixels,
//          blended front to back in draw order with the reference's blend
//          state (colour = src*DstAlpha + dst, alpha = dst*(1-srcA), cleared
//          to (0,0,0,1)), the unorm8 target emulated by clamping the source
//          and re-quantising after every blend; a wave stops once its pixels'
//          transmittance is 0, a tile once all four have.  The tiles with the
//          longest lists get blocks of their own (raster_heavy.h).
#include "raster_common.h"
#include "raster_heavy.h"

namespace spl {

namespace {

// Per-lane walk over one run of cnt <= 32 entries (cm, ct, cc: their three
// staged rows, in list order, in LDS) of a wave's 8x8 region with top-left
// pixel (fqx0, fqy0); rows: 64 words of LDS for the coverage rows.  The wave
// first finds, for every pixel, the run's entries that can cover it, then
// every lane walks only those, in list order, each lane on its own: the
// wave takes as many steps as its busiest pixel has covering entries, not
// as many as the run has.
//
// The candidates come per row, entry-parallel: 2, 4 or 8 lanes per entry
// each take 4, 2 or 1 of the region's rows and solve the rectangle's two
// slabs |a px + b py + c| < h for the row's column interval, widened by far
// more than the rounding of either that solution or the per-pixel test
// (2^-19 of the magnitudes, against about 12 roundings of 2^-24), so it
// holds every column whose centre the per-pixel test accepts.  A slab that
// hardly varies along x (|a| < h 1e-6), or with a coefficient that is not
// finite, is taken as all columns.  Each pixel lane then gathers its row's
// 32 bits from LDS (row y: byte 3 - (k >> 3) of word k & 7 holds slot k's
// row mask, bit x = column x), and the walk applies the exact per-pixel
// test of the other modes to every candidate (a candidate that fails it
// blends with alpha 0, which leaves the pixel as it is), so the pixels are
// the same.  Runs of up to 12 entries are tested per pixel instead.
template <bool UNALIGNED, bool F32>
__device__ __forceinline__ void walk_run(const float4* cm, const float4* ct, const float4* cc, uint32_t* rows,
                                         uint32_t cnt, uint32_t lane, bool inside, float pxf, float pyf, float fqx0,
                                         float fqy0, float span, const PixelMap& pm, float margin,
                                         PixelState<F32>& pix) {
  uint8_t* const rows8 = reinterpret_cast<uint8_t*>(rows);
  constexpr uint32_t kRowsMin = 12;  // runs up to this long are tested per pixel
  // column interval of row y (local, 0..7) as [ceil(lo), floor(hi1) - 1],
  // clamped to the region, as a row mask
  auto row_mask = [&](float lo, float hi1) -> uint32_t {
    const uint32_t first = (uint32_t)__builtin_amdgcn_fmed3f(ceilf(lo), 0.0f, 8.0f);
    const uint32_t end = (uint32_t)__builtin_amdgcn_fmed3f(floorf(hi1), 0.0f, 8.0f);
    return ((1u << end) - 1u) & ~((1u << first) - 1u);
  };
  // slab |a px + b py + c| < h in local columns: lo(y) = P y + lo0,
  // hi(y) + 1 = P y + hi0
  auto slab = [&](float a_, float b_, float c_, float h_, float& P, float& lo0, float& hi0) {
    const float ia = __builtin_amdgcn_rcpf(a_);
    const float R = h_ * fabsf(ia);
    const float Pv = -b_ * ia;
    const float Qg = -c_ * ia;
    const float Q = fmaf(Pv, fqy0, Qg) - fqx0;
    const float eps = 0x1p-19f * (((fabsf(Pv) * span + fabsf(Qg)) + R) + span) + 0x1p-19f;
    // (R = 0 for an infinite a, whose products with a zero
    // coordinate are NaN in the per-pixel test)
    const bool ok = R > 0.0f && R < 1e6f && fabsf(Pv) < 1e6f && fabsf(Qg) < 1e9f;
    P = ok ? Pv : 0.0f;
    lo0 = ok ? (Q - R) - eps : -1e9f;
    hi0 = ok ? ((Q + R) + eps) + 1.0f : 1e9f;
  };
  uint32_t mask = 0;
  if (cnt <= kRowsMin) {
    // a short run: every lane tests its pixel against each slot
    // (exact), slot k at bit K - 1 - k for K = cnt rounded up to 4
    for (uint32_t k = 0; k < cnt; k += 4) {
      uint32_t nib = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float u, w2;
        float4 t4;
        if constexpr (UNALIGNED) {
          // the half-extent is margin * S for every entry
          const float2 t2 = *reinterpret_cast<const float2*>(&ct[k + q]);
          t4 = make_float4(t2.x, t2.y, margin * kGaussScale, 0.0f);
        } else {
          t4 = ct[k + q];
        }
        nib = (nib << 1) | (covers<UNALIGNED>(cm[k + q], t4, pxf, pyf, pm, u, w2) ? 1u : 0u);
      }
      mask = (mask << 4) | nib;
    }
    mask <<= 32u - ((cnt + 3u) & ~3u);
  } else {
    {
      const uint32_t lpe = cnt <= 8u ? 3u : (cnt <= 16u ? 2u : 1u);  // log2 lanes per entry
      const uint32_t k = lane >> lpe;
      if (k < cnt) {
        const uint32_t rpl = 8u >> lpe;  // rows per lane
        const uint32_t y0 = (lane & ((1u << lpe) - 1u)) * rpl;
        const float4 m = cm[k];
        const float4 t = ct[k];
        uint8_t* const dst = rows8 + (k & 7u) * 4u + (3u - (k >> 3));
        if constexpr (UNALIGNED) {
          const float h = margin * kGaussScale;
          float P1, l1, e1, P2, l2, e2;
          slab(m.x, m.y, t.x, h, P1, l1, e1);
          slab(m.z, m.w, t.y, h, P2, l2, e2);
          for (uint32_t i = 0; i < rpl; ++i) {
            const float y = (float)(y0 + i);
            const float lo = fmaxf(fmaf(P1, y, l1), fmaf(P2, y, l2));
            const float hi1 = fminf(fmaf(P1, y, e1), fmaf(P2, y, e2));
            dst[(y0 + i) * 32u] = (uint8_t)row_mask(lo, hi1);
          }
        } else {
          // dx = sx px + t.x bounds the columns, dy = sy py + t.y the rows
          float P, lx, ex, Py, ly, ey;
          slab(pm.sx, 0.0f, t.x, t.z, P, lx, ex);
          slab(pm.sy, 0.0f, t.y, t.z, Py, ly, ey);
          // rows: the same interval, in rows (py in place of px)
          ly += fqx0 - fqy0;
          ey += fqx0 - fqy0;
          const uint32_t cols = row_mask(lx, ex);
          const uint32_t rmask = row_mask(ly, ey);
          for (uint32_t i = 0; i < rpl; ++i)
            dst[(y0 + i) * 32u] = (uint8_t)(((rmask >> (y0 + i)) & 1u) ? cols : 0u);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
    // this pixel's candidates: slot k at bit 31 - k
    const uint32_t xl = lane & 7u;
    const uint4 ra = *reinterpret_cast<const uint4*>(&rows[(lane >> 3) * 8u]);
    const uint4 rb = *reinterpret_cast<const uint4*>(&rows[(lane >> 3) * 8u + 4u]);
    mask = (mask << 1) | ((ra.x >> xl) & 0x01010101u);
    mask = (mask << 1) | ((ra.y >> xl) & 0x01010101u);
    mask = (mask << 1) | ((ra.z >> xl) & 0x01010101u);
    mask = (mask << 1) | ((ra.w >> xl) & 0x01010101u);
    mask = (mask << 1) | ((rb.x >> xl) & 0x01010101u);
    mask = (mask << 1) | ((rb.y >> xl) & 0x01010101u);
    mask = (mask << 1) | ((rb.z >> xl) & 0x01010101u);
    mask = (mask << 1) | ((rb.w >> xl) & 0x01010101u);
  }
  mask &= ~0u << (32u - cnt);  // slots at or past cnt hold stale rows
  if (pix.tr == 0.0f || !inside) mask = 0u;
  while (mask) {
    const uint32_t k = (uint32_t)__builtin_clz(mask);
    mask &= ~(0x80000000u >> k);
    const float4 t = ct[k];
    float u, w2;
    const bool in = covers<UNALIGNED>(cm[k], t, pxf, pyf, pm, u, w2);
    pix.shade(u, w2, t.w, cc[k], in);
    if (pix.tr == 0.0f) mask = 0u;
  }
}

}  // namespace

// Bound by the latency of a tile's chain (ticket, box gather, look-back) in
// small frames and by the expansion's LDS reads and VALU in large ones.  Each
// entry of the tile is one 16-byte LDS row (first output slot, first screen
// tile and width packed, record), stored item-major so that a wave writes
// consecutive rows; logical entry i = 4 tid + k (ITEMS = 4) is row
// k * THREADS + tid.  Tiles of more than 4096 pairs expand through the owner
// table 4096 slots at a time (a binary search over the offsets, ten dependent
// LDS reads a pair, took 61 us on 100k splats at 720p, which take 16 now; 8
// views of 32M at 4K render in 65.7 ms instead of 70.5).
template <int THREADS, int ITEMS>
__global__ __launch_bounds__(THREADS) void k_bin(BinLaunch a) {
  constexpr int TILE = THREADS * ITEMS;
  constexpr int WAVES = THREADS / kWave;
  constexpr int REP = 2;  // histogram copies across lanes: neighbouring pairs share their high digit
  __shared__ uint4 s_ent[TILE];
  // the entry that owns each of OWN output slots
  constexpr uint32_t OWN = 4096, PER = OWN / THREADS;
  static_assert(PER == 16, "a thread's owner slots are two 16-byte LDS rows");
  __shared__ __align__(16) uint16_t s_own[OWN];
  __shared__ uint32_t s_hist[kMaxPairPasses * 256 * REP];
  __shared__ uint32_t s_tmp[WAVES];
  __shared__ uint32_t s_tile;
  __shared__ uint64_t s_prefix;

  const uint32_t tid = threadIdx.x;
  const uint32_t v = blockIdx.y;
  uint32_t* counters = a.counters + (size_t)v * kCounterWords;
  const uint32_t* order = a.order ? a.order + v * a.order_stride : nullptr;
  const uint2* boxes = a.boxes + v * a.box_stride;
  uint32_t* pair_keys = a.pair_keys + v * a.pair_stride;
  uint32_t* pair_vals = a.pair_vals + v * a.pair_stride;
  uint64_t* status = a.status + v * a.status_stride;
  if (a.clear_a) clear_words(a.clear_a + v * a.clear_a_stride, a.clear_a_words);
  if (a.clear_b) clear_words(a.clear_b + v * a.clear_b_stride, a.clear_b_words);
  for (int i = tid; i < a.pair_passes * 256 * REP; i += THREADS) s_hist[i] = 0u;
  const uint32_t n = counters[kVisible];
  const uint32_t num_tiles = (n + TILE - 1) / TILE;
  if (num_tiles == 0 && blockIdx.x == 0 && tid == 0) {
    counters[kPairs] = 0u;
    counters[kPairOverflow] = 0u;
  }
  if (persistent_idle(num_tiles)) return;
  const uint32_t tiles_x = a.uniforms[v].tiles_x;

  while (true) {
    if (tid == 0) s_tile = take_ticket(&counters[kCtrBin], num_tiles);
    __syncthreads();
    const uint32_t t = s_tile;
    if (t >= num_tiles) break;
    // The items' record indices, then their boxes, are all requested before
    // any is used (past the end a lane reads item 0 and drops it), so that
    // no load waits for the one before.
    uint32_t cnt[ITEMS], sum = 0, rec[ITEMS];
    uint2 box[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      const uint32_t r = t * TILE + tid * ITEMS + k;
      rec[k] = order ? order[r < n ? r : 0u] : r;
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      const uint32_t r = t * TILE + tid * ITEMS + k;
      if (r < n && rec[k] >= n) counters[kScatterError] = 1u;  // only after an upstream error
      if (r >= n || rec[k] >= n) rec[k] = 0u;  // never read past the boxes
      box[k] = boxes[rec[k]];
    }
    // screen tiles up to 1024 across and down (frames up to 16384 pixels):
    // x, y and the width of at most 1024 pack into 31 bits
    static_assert(kTileSize == 16, "tile coordinates in 10 bits");
    uint32_t geom[ITEMS], off[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      const uint32_t r = t * TILE + tid * ITEMS + k;
      cnt[k] = 0;
      geom[k] = 1u << 20;
      if (r < n) {
        const uint2 q = box[k];
        const uint32_t lo = q.x, hi = q.y;
        const uint32_t x0 = (lo & 0xFFFFu) / kTileSize, y0 = (lo >> 16) / kTileSize;
        const uint32_t x1 = (hi & 0xFFFFu) / kTileSize, y1 = (hi >> 16) / kTileSize;
        if (lo != 0xFFFFFFFFu && x1 >= x0 && y1 >= y0) {
          cnt[k] = (x1 - x0 + 1) * (y1 - y0 + 1);
          geom[k] = x0 | (y0 << 10) | ((x1 - x0 + 1) << 20);
        }
      }
      sum += cnt[k];
    }
    uint32_t total;
    uint32_t excl = block_exclusive_scan<THREADS>(sum, s_tmp, total);
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      off[k] = excl;
      s_ent[k * THREADS + tid] = make_uint4(excl, geom[k], rec[k], 0u);
      excl += cnt[k];
    }
    if (tid < kWave) {
      const uint64_t prefix = wave_lookback64(status, t, (uint64_t)total);
      if (tid == 0) s_prefix = prefix;
      if (tid == 0 && t == num_tiles - 1) {
        const uint64_t k_all = prefix + total;
        counters[kPairs] = (uint32_t)(k_all < a.pair_cap ? k_all : a.pair_cap);
        counters[kPairOverflow] = k_all > a.pair_cap ? 1u : 0u;
      }
    }
    // Output slots, OWN at a time.  Owner of each: every entry with pairs in
    // them writes its index at its first, then an inclusive max-scan carries
    // the indices forward.  (Slots past the last hold stale owners: the scan
    // carries them only forward, into slots that no pair reads.)
    const uint32_t lane = tid & (kWave - 1), wv = tid / kWave;
    uint4* const own4 = reinterpret_cast<uint4*>(s_own);  // eight slots a row
    for (uint32_t s0 = 0; s0 < total; s0 += OWN) {
      const uint32_t m = min(total - s0, OWN);
      for (uint32_t q = tid; q < (m + 7u) / 8u; q += THREADS) own4[q] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < ITEMS; ++k)
        if (cnt[k] > 0u && off[k] + cnt[k] > s0 && off[k] < s0 + OWN)
          s_own[max(off[k], s0) - s0] = (uint16_t)(tid * ITEMS + k);
      __syncthreads();
      // this thread's sixteen slots, two rows; slot 2i + h is half h of word i
      const uint4 ra = own4[2 * tid], rb = own4[2 * tid + 1];
      uint32_t wd[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
      uint32_t run = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) run = max(run, max(wd[i] & 0xFFFFu, wd[i] >> 16));
      uint32_t incl = run;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o, kWave);
        if (lane >= (uint32_t)o) incl = max(incl, y);
      }
      if (lane == kWave - 1) s_tmp[wv] = incl;
      __syncthreads();
      uint32_t carry = __shfl_up(incl, 1, kWave);
      if (lane == 0) carry = 0;
      for (uint32_t i = 0; i < wv; ++i) carry = max(carry, s_tmp[i]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t lo = max(carry, wd[i] & 0xFFFFu);
        carry = max(lo, wd[i] >> 16);
        wd[i] = lo | (carry << 16);
      }
      own4[2 * tid] = make_uint4(wd[0], wd[1], wd[2], wd[3]);
      own4[2 * tid + 1] = make_uint4(wd[4], wd[5], wd[6], wd[7]);
      __syncthreads();
      const uint64_t prefix = s_prefix + s0;
      for (uint32_t s = tid; s < m; s += THREADS) {
        const uint32_t lo = s_own[s];
        const uint4 e = s_ent[lo % ITEMS * THREADS + lo / ITEMS];
        const uint64_t pos = prefix + s;
        if (pos < a.pair_cap) {
          // row and column of pair k in a box w tiles wide: (k + 1/2) / w is
          // at least 1/2w from an integer, and the product's error is below
          // (k + 1/2) / w * 2^-22, so its floor is k / w for k < 2^20
          const uint32_t k = s0 + s - e.x, w = e.y >> 20;
          const uint32_t row = (uint32_t)(((float)k + 0.5f) * __builtin_amdgcn_rcpf((float)w));
          const uint32_t tile = (((e.y >> 10) & 1023u) + row) * tiles_x + (e.y & 1023u) + (k - row * w);
          pair_keys[pos] = tile;
          pair_vals[pos] = e.z;
          for (int q = 0; q < a.pair_passes; ++q)
            atomicAdd(&s_hist[(q * 256 + ((tile >> (8 * q)) & 255u)) * REP + (tid & (REP - 1))], 1u);
        }
      }
      __syncthreads();
    }
    if (one_tile_each(num_tiles)) break;
    __syncthreads();
  }
  __syncthreads();
  // each XCD's blocks add to a copy of their own: an address that every block
  // adds to takes 11.5 ns a block
  uint32_t* hist = a.hist + v * a.hist_stride + (blockIdx.x % kHistCopies) * (kMaxPairPasses * 256);
  for (int i = tid; i < a.pair_passes * 256; i += THREADS) {
    uint32_t c = 0;
#pragma unroll
    for (int r = 0; r < REP; ++r) c += s_hist[i * REP + r];
    if (c) atomicAdd(&hist[i], c);
  }
}

// Run boundaries of the tile-sorted pair keys, four keys per thread.
__global__ __launch_bounds__(256) void k_tile_ranges(RangesLaunch a) {
  const uint32_t v = blockIdx.y;
  if (a.clear_a)
    clear_words(a.clear_a + v * a.clear_a_stride,
                used_status(a.clear_a_words, a.clear_a_tile, a.one_round, a.counters[(size_t)v * kCounterWords + kPairs]));
  if (a.clear_b) clear_words(a.clear_b + v * a.clear_b_stride, a.clear_b_words);
  if (blockIdx.x == 0 && v == 0 && threadIdx.x <= kHeavyClasses + 1) a.counters[kHeavyAll + threadIdx.x] = 0u;
  const uint32_t* keys = a.pair_keys + v * a.pair_stride;  // 16-byte aligned: pair_stride % 4 == 0
  uint2* ranges = a.ranges + v * a.ranges_stride;
  const uint32_t tiles = a.uniforms[v].tiles_x * a.uniforms[v].tiles_y;
  uint32_t n = a.counters[(size_t)v * kCounterWords + kPairs];
  if (n > a.pair_cap) n = a.pair_cap;
  const uint32_t step = gridDim.x * blockDim.x * 4;
  for (uint32_t i0 = (blockIdx.x * blockDim.x + threadIdx.x) * 4; i0 < n; i0 += step) {
    // the three loads go out together: out of range they read key 0 (or
    // the run's first key) and the value is replaced after
    uint32_t k[6];
    const uint32_t prev = keys[i0 > 0 ? i0 - 1 : 0u];
    const uint32_t next = keys[i0 + 4 < n ? i0 + 4 : 0u];
    if (i0 + 4 <= n) {
      const uint4 q = *reinterpret_cast<const uint4*>(keys + i0);
      k[1] = q.x; k[2] = q.y; k[3] = q.z; k[4] = q.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) k[1 + j] = i0 + j < n ? keys[i0 + j] : 0xFFFFFFFFu;
    }
    k[0] = i0 > 0 ? prev : 0xFFFFFFFFu;
    k[5] = i0 + 4 < n ? next : 0xFFFFFFFFu;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t i = i0 + j, t = k[1 + j];
      if (i >= n || t >= tiles) continue;
      if (k[j] != t) ranges[t].x = i;
      if (k[2 + j] != t) ranges[t].y = i + 1;
    }
  }
}

// The tiles whose lists are long enough to set the raster's time by
// themselves ("heavy", kHeavyShare has the rule).  k_raster gives each eight
// blocks, longest first: they are listed by length in kHeavyClasses lists (the
// last for 16 x the threshold and more), and the top bit of a listed tile's
// range start tells its ordinary block to leave it alone.  One thread per
// tile; appends are atomics on counters that k_tile_ranges zeroed.  (The one
// block that put the tiles in order before took 14 us at 1080p and 65 at 4K;
// this takes 4 to 8.)
__global__ __launch_bounds__(256) void k_heavy_tiles(HeavyLaunch a) {
  const uint32_t v = blockIdx.y, t = blockIdx.x * 256 + threadIdx.x;
  const uint32_t T = a.uniforms[v].tiles_x * a.uniforms[v].tiles_y;
  if (t >= T) return;
  uint64_t pairs = 0;
  for (int i = 0; i < a.views; ++i) pairs += min(a.counters[(size_t)i * kCounterWords + kPairs], a.pair_cap);
  const uint32_t thr = max((uint32_t)min(pairs / kHeavyShare, (uint64_t)0x40000000u), kHeavyMin);
  uint2* range = a.ranges + v * a.ranges_stride + t;
  const uint2 r = *range;
  const uint32_t len = r.y - r.x;
  if (len < thr) {
    // a long tile among the ordinary ones starts ahead of them
    const uint32_t mine = min(a.counters[(size_t)v * kCounterWords + kPairs], a.pair_cap);
    if (len < max(thr / 4u, 2u * (mine / T))) return;
    const uint32_t at = atomicAdd(&a.counters[kLongTiles], 1u);
    if (at >= a.long_cap) return;
    a.list[kHeavyClasses * kHeavyCap + at] = (v << 24) | t;
    range->x = r.x | kHeavyFlag;
    return;
  }
  const uint32_t times = len / thr;
  const uint32_t c = times >= 16u ? 3u : times >= 4u ? 2u : times >= 2u ? 1u : 0u;
  uint32_t* const all = a.counters;  // one set of lists for all views, counted in view 0's block
  if (atomicAdd(&all[kHeavyAll], 1u) >= a.heavy_cap) return;
  const uint32_t at = atomicAdd(&all[kHeavyTiles + c], 1u);
  a.list[c * kHeavyCap + at] = (v << 24) | t;
  range->x = r.x | kHeavyFlag;
  if (a.tile_work && v == 0) a.tile_work[t] = make_uint2(len, 0u);
}

void launch_heavy_tiles(const HeavyLaunch& a, hipStream_t s) {
  hipLaunchKernelGGL(k_heavy_tiles, dim3((a.max_tiles + 255) / 256, a.views), dim3(256), 0, s, a);
}

// One 256-lane block per 16x16 tile; wave w owns the 8x8 quadrant
// (w & 1, w >> 1), one lane per pixel.  Entries arrive B at a time in draw
// order: every lane gathers one record and stores the prepared entry (inverse
// affine map, translation, coverage half-extent, colour, pixel box) in LDS,
// while the next batch is already being fetched into registers.  Each wave
// then keeps, in order, only the entries whose pixel box meets its quadrant
// (ballot + mbcnt) and blends those; a wave whose 64 pixels are all opaque
// stops blending, and the block stops when all four have.
template <bool UNALIGNED, bool F32, int MODE, int B>
// (mode 3 occupancy: 128-entry batches at seven waves per SIMD, 72 VGPRs, none
// spilled; the f32 blend needs 78 or 79 and keeps six; 256-entry batches need
// 84 to 86, and 31 KB of LDS, and run five)
__global__ __launch_bounds__(256, MODE == 3 ? (B == 128 ? (F32 ? 6 : 7) : 5) : 1) void k_raster(RasterLaunch a) {
  static_assert(B == 128 || B == 256, "entries staged per batch");
  constexpr int U = B / 64;  // list slots per step of the entry-major walks
  constexpr bool WALK = MODE == 1, SUBS = MODE == 2, LANES = MODE == 3;
  constexpr bool LANES_ = LANES;
  // per staged entry: [0] i00 i01 i10 i11, [1] tx ty half alpha, [2] r g b -
  // (one array, so an entry's three rows share one LDS address)
  __shared__ float4 s_ent[2][3][B];
  __shared__ uint2 s_box[2][B];    // pixel box lo / hi (x | y << 16)
  __shared__ __align__(16) uint8_t s_list[4][B];  // per-wave compacted entry slots, read 4 at a time
  // mode 3: per wave, the coverage of 32 run slots as 8 rows x 8 words; byte
  // 3 - (k >> 3) of word k & 7 of row y holds slot k's row mask (bit x =
  // column x of the quadrant)
  __shared__ __align__(16) uint32_t s_rows[LANES_ ? 4 : 1][LANES_ ? 64 : 4];
  __shared__ __align__(16) uint8_t s_sub[SUBS ? 4 : 1][SUBS ? 4 : 1][SUBS ? B : 4];  // mode 2: per 4x4 sub-block

  // Block -> (view, tile).  First eight blocks for each heavy tile, longest
  // class first, then one for each long tile, then each view's tiles in a slot
  // range of slots_per_view blocks.  Blocks are dealt round-robin to the 8 XCDs, and the XCDs take
  // runs of kXcdRun neighbouring tiles in turn (kXcdRun has why).
  uint32_t b = blockIdx.x;
  const uint32_t heavy = min(a.counters[kHeavyAll], a.heavy_cap), heavy_blocks = 8u * ((heavy + 7u) & ~7u);
  if (b < heavy_blocks) {
    __shared__ __align__(16) uint32_t s_words[8];
    // a tile's blocks on one XCD: they read the same records
    uint32_t at = b / 64u * 8u + (b & 7u);
    if (at >= heavy) return;
    int c = kHeavyClasses - 1;
    for (; c > 0; --c) {
      const uint32_t h = a.counters[kHeavyTiles + c];
      if (at < h) break;
      at -= h;
    }
    const uint32_t vt = a.heavy[c * kHeavyCap + at];
    raster_heavy<UNALIGNED, F32>(a, vt >> 24, vt & 0xFFFFFFu, (b >> 3) & 7u, &s_ent[0][0][0], s_words);
    return;
  }
  b -= heavy_blocks;
  uint32_t v, tile;
  const uint32_t longs = min(a.counters[kLongTiles], a.long_cap), long_blocks = (longs + 7u) & ~7u;
  const bool listed = b < long_blocks;
  if (listed) {
    if (b >= longs) return;
    const uint32_t vt = a.heavy[kHeavyClasses * kHeavyCap + b];
    v = vt >> 24;
    tile = vt & 0xFFFFFFu;
  } else {
    b -= long_blocks;
    v = b / a.slots_per_view;
    if (v >= (uint32_t)a.views) return;
    const uint32_t slot = b % a.slots_per_view;
    tile = ((slot >> 3) / kXcdRun * 8u + (slot & 7u)) * kXcdRun + (slot >> 3) % kXcdRun;
    if (tile >= a.uniforms[v].tiles_x * a.uniforms[v].tiles_y) return;
  }
  const Uniforms& u = a.uniforms[v];
  const uint2* ranges = a.ranges + v * a.ranges_stride;
  const uint32_t* pair_vals = a.pair_vals + v * a.pair_stride;
  const float4* records = a.records + v * a.rec_stride;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  // this wave's 8x8 region: quadrant w
  const uint32_t qx0 = (tile % u.tiles_x) * kTileSize + (w & 1u) * 8u;
  const uint32_t qy0 = (tile / u.tiles_x) * kTileSize + (w >> 1) * 8u;
  // mode 2: lane group g = lane / 16 owns the 4x4 sub-block (g & 1, g >> 1)
  const uint32_t g = lane >> 4;
  const uint32_t px = SUBS ? qx0 + (g & 1u) * 4u + (lane & 3u) : qx0 + (lane & 7u);
  const uint32_t py = SUBS ? qy0 + (g >> 1) * 4u + ((lane >> 2) & 3u) : qy0 + (lane >> 3);
  const uint32_t W = u.image_size[0], H = u.image_size[1];
  const bool inside = px < W && py < H;
  // (the ranges are cleared for the next frame by its pair sort)
  uint2 range = ranges[tile];
  if (listed) range.x &= ~kHeavyFlag;
  else if (range.x & kHeavyFlag) return;  // has blocks of its own

  const PixelMap pm = pixel_map(u);
  const float pxf = (float)px, pyf = (float)py;
  const float margin = u.ellipse_margin;
  PixelState<F32> pix;
  const uint32_t visible = a.counters[(size_t)v * kCounterWords + kVisible];

  // register stage of one entry per lane
  float4 g0 = make_float4(0, 0, 0, 0), g1 = g0, g2 = g0;
  auto fetch = [&](uint32_t base) {
    if (tid < (uint32_t)B && base + tid < range.y) {
      uint32_t c = pair_vals[base + tid];
      if (c >= visible) c = 0;  // only after an upstream error; never read past the records
      g0 = records[3 * (size_t)c + 0];
      g1 = records[3 * (size_t)c + 1];
      g2 = records[3 * (size_t)c + 2];
    }
  };
  auto stage = [&](int buf) {
    if (tid >= (uint32_t)B) return;
    prepare_entry<UNALIGNED>(g0, g1, g2, pm, margin, s_ent[buf][0][tid], s_ent[buf][1][tid], s_ent[buf][2][tid]);
    s_box[buf][tid] = make_uint2(__float_as_uint(g2.z), __float_as_uint(g2.w));
  };

  // lanes whose pixel still takes fragments (inside the image, not yet
  // opaque); in modes 0 and 1 lane y * 8 + x holds pixel (x, y) of the quadrant
  uint64_t alive = __ballot(inside);
  bool wave_done = alive == 0ull;
  uint32_t consumed = 0;
  int buf = 0;
  if (range.x < range.y) {
    fetch(range.x);
    stage(0);
  }
  __syncthreads();
  for (uint32_t base = range.x; base < range.y; base += B) {
    const uint32_t cnt = (range.y - base) < (uint32_t)B ? (range.y - base) : (uint32_t)B;
    const bool more = base + B < range.y;
    if (more) fetch(base + B);
    consumed += cnt;
    if (!wave_done) {
      // Entries of this batch that can cover a pixel centre still taking
      // fragments, in order: pixel box against the box of the live pixels,
      // then the exact range of the coverage coordinate over that box's
      // pixel centres (it is affine in the centre, so its extremes sit at the
      // corner centres).  An entry that meets only opaque pixels would add
      // s * 0 to them, so leaving it out changes nothing.  The live box's
      // columns come from the OR of the mask's eight rows, its rows from the
      // lowest and highest set bits.  Mode 2 lays its lanes out per sub-block
      // (bits 16 g .. 16 g + 15 are sub-block g): it keeps the quadrant's box
      // and skips opaque sub-blocks instead.
      uint32_t ax0 = qx0, ax1 = min(qx0 + 7u, W - 1u), ay0 = qy0, ay1 = min(qy0 + 7u, H - 1u);
      if constexpr (!SUBS) {
        uint32_t cols = (uint32_t)alive | (uint32_t)(alive >> 32);
        cols |= cols >> 16;
        cols |= cols >> 8;
        ax0 = qx0 + (uint32_t)__builtin_ctz(cols & 0xFFu);
        ax1 = qx0 + 31u - (uint32_t)__builtin_clz(cols & 0xFFu);
        ay0 = qy0 + ((uint32_t)__builtin_ctzll(alive) >> 3);
        ay1 = qy0 + ((63u - (uint32_t)__builtin_clzll(alive)) >> 3);
      }
      uint32_t n = 0;
      uint32_t ns[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int k = 0; k < B / 64; ++k) {
        const uint32_t j = k * 64 + lane;
        bool ov = false;
        if (j < cnt) {
          const uint2 bx = s_box[buf][j];
          const uint32_t x0 = bx.x & 0xFFFFu, y0 = bx.x >> 16, x1 = bx.y & 0xFFFFu, y1 = bx.y >> 16;
          ov = bx.x != 0xFFFFFFFFu && x0 <= ax1 && x1 >= ax0 && y0 <= ay1 && y1 >= ay0;
          if (ov && !SUBS)
            ov = range_meets<UNALIGNED>(s_ent[buf][0][j], s_ent[buf][1][j], (float)ax0, (float)ax1, (float)ay0,
                                        (float)ay1, pm);
        }
        if constexpr (!SUBS) {
          const uint64_t bm = __ballot(ov);
          if (ov) s_list[w][n + lanes_below(bm)] = (uint8_t)j;
          n += (uint32_t)__popcll(bm);
        } else {
          // the same exact test per 4x4 sub-block, one list each
#pragma unroll
          for (int sb = 0; sb < 4; ++sb) {
            // a sub-block whose pixels are all opaque takes no entries
            bool o = ov && ((alive >> (16 * sb)) & 0xFFFFull) != 0ull;
            if (o) {
              const uint32_t bx0 = qx0 + (sb & 1) * 4u, by0 = qy0 + (sb >> 1) * 4u;
              const uint2 bx = s_box[buf][j];
              o = bx0 < W && by0 < H && (bx.x & 0xFFFFu) <= bx0 + 3u && (bx.y & 0xFFFFu) >= bx0 &&
                  (bx.x >> 16) <= by0 + 3u && (bx.y >> 16) >= by0;
              if (o) {
                const uint32_t bx1 = min(bx0 + 3u, W - 1u), by1 = min(by0 + 3u, H - 1u);
                o = range_meets<UNALIGNED>(s_ent[buf][0][j], s_ent[buf][1][j], (float)bx0, (float)bx1, (float)by0,
                                           (float)by1, pm);
              }
            }
            const uint64_t bm = __ballot(o);
            if (o) s_sub[w][sb][ns[sb] + lanes_below(bm)] = (uint8_t)j;
            ns[sb] += (uint32_t)__popcll(bm);
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
      // one fragment at this lane's pixel: coverage, alpha (shaders.wgsl:585-589)
      // and the blend; identical arithmetic on every walk, so they give
      // identical pixels
      auto covers_ = [&](const float4& m, const float4& t, float& u, float& w2) -> bool {
        return covers<UNALIGNED>(m, t, pxf, pyf, pm, u, w2);
      };
      auto shade = [&](float u, float w2, float opacity, const float4& col, bool in) {
        pix.shade(u, w2, opacity, col, in);
      };
      if constexpr (SUBS) {
        // entry-major per 4x4 sub-block: the four lane groups step through
        // their own lists side by side, so one step blends up to four entries
        const uint32_t mine = g == 0 ? ns[0] : g == 1 ? ns[1] : g == 2 ? ns[2] : ns[3];
        const uint32_t most = max(max(ns[0], ns[1]), max(ns[2], ns[3]));
        for (uint32_t i = 0; i < most; i += U) {
          uint32_t js;
          if constexpr (U == 4) js = *reinterpret_cast<const uint32_t*>(&s_sub[w][g][i]);
          else js = *reinterpret_cast<const uint16_t*>(&s_sub[w][g][i]);
          float4 m[U], t[U], col[U];
#pragma unroll
          for (int k = 0; k < U; ++k) {
            // slots past the list may be stale or, on a block's first batch,
            // uninitialised: masked into [0, B) they still index s_ent, and
            // their fragments are never blended (i + k < mine)
            const uint32_t j = (js >> (8 * k)) & (uint32_t)(B - 1);
            m[k] = s_ent[buf][0][j];
            t[k] = s_ent[buf][1][j];
            col[k] = s_ent[buf][2][j];
          }
#pragma unroll
          for (int k = 0; k < U; ++k) {
            float u, w2;
            if (i + k < mine && covers_(m[k], t[k], u, w2) && pix.tr != 0.0f) shade(u, w2, t[k].w, col[k], true);
          }
        }
      } else if constexpr (LANES) {
        // per-lane walk: for 32 list slots at a time the wave first copies
        // the slots' entries into a compact run (its 32 entries of the
        // other staging buffer, free until the next batch is staged), then
        // walks the run (walk_run: each pixel only its covering entries)
        float4* const cm = &s_ent[buf ^ 1][0][32 * w];
        float4* const ct = &s_ent[buf ^ 1][1][32 * w];
        float4* const cc = &s_ent[buf ^ 1][2][32 * w];
        const float fqx0 = (float)qx0, fqy0 = (float)qy0;
        const float span = (float)W + (float)H;  // bounds the pixel coordinates' magnitudes
        for (uint32_t c = 0; c < n; c += 32) {
          const uint32_t cnt = min(32u, n - c);
          if (lane < cnt) {
            const uint32_t j = (uint32_t)s_list[w][c + lane] & (uint32_t)(B - 1);
            cm[lane] = s_ent[buf][0][j];
            ct[lane] = s_ent[buf][1][j];
            cc[lane] = s_ent[buf][2][j];
          }
          __builtin_amdgcn_wave_barrier();
          walk_run<UNALIGNED, F32>(cm, ct, cc, &s_rows[w][0], cnt, lane, inside, pxf, pyf, fqx0, fqy0, span, pm,
                                   margin, pix);
          __builtin_amdgcn_wave_barrier();
        }
      } else if constexpr (!WALK) {
        // entry-major: the wave steps through its list, every lane testing
        // its pixel; four list slots per step so their LDS reads go together
        for (uint32_t i = 0; i < n; i += U) {
          uint32_t js;
          if constexpr (U == 4) js = *reinterpret_cast<const uint32_t*>(&s_list[w][i]);
          else js = *reinterpret_cast<const uint16_t*>(&s_list[w][i]);
          float4 m[U], t[U], col[U];
#pragma unroll
          for (int k = 0; k < U; ++k) {
            // slots past n may be stale or, on a block's first batch,
            // uninitialised: masked into [0, B) they still index s_ent, and
            // the loop below stops at n before using them
            const uint32_t j = (js >> (8 * k)) & (uint32_t)(B - 1);
            m[k] = s_ent[buf][0][j];
            t[k] = s_ent[buf][1][j];
            col[k] = s_ent[buf][2][j];
          }
#pragma unroll
          for (int k = 0; k < U; ++k) {
            if (i + k >= n) break;
            float u, w2;
            if (covers_(m[k], t[k], u, w2) && pix.tr != 0.0f) shade(u, w2, t[k].w, col[k], true);
          }
        }
      } else {
        // pixel-major: for 64 list slots at a time every lane first marks the
        // entries that cover its pixel, then walks only those, in order, so
        // lanes are not held up by entries that cover few of the 64 pixels
        for (uint32_t c = 0; c < n; c += 64) {
          const uint32_t cnt = min(64u, n - c);
          uint32_t lo = 0, hi = 0;
          for (uint32_t k = 0; k < cnt; k += 4) {
            const uint32_t js = *reinterpret_cast<const uint32_t*>(&s_list[w][c + k]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const uint32_t j = (js >> (8 * q)) & 255u;
              float u, w2;
              const uint32_t in = covers_(s_ent[buf][0][j], s_ent[buf][1][j], u, w2) && k + q < cnt ? 1u : 0u;
              if (k < 32) lo |= in << (k + q);
              else hi |= in << (k + q - 32);
            }
          }
          if (pix.tr == 0.0f) lo = hi = 0u;
          while (lo | hi) {
            uint32_t k;
            if (lo) { k = (uint32_t)__builtin_ctz(lo); lo &= lo - 1u; }
            else { k = 32u + (uint32_t)__builtin_ctz(hi); hi &= hi - 1u; }
            const uint32_t j = s_list[w][c + k];
            const float4 t = s_ent[buf][1][j];
            float u, w2;
            (void)covers_(s_ent[buf][0][j], t, u, w2);
            shade(u, w2, t.w, s_ent[buf][2][j], true);
            if (pix.tr == 0.0f) lo = hi = 0u;
          }
        }
      }
      alive = __ballot(inside && pix.tr != 0.0f);
      wave_done = alive == 0ull;
    }
    if (more) {
      // mode 3's compact runs live in the other buffer until every wave has
      // walked
      if constexpr (LANES) __syncthreads();
      stage(buf ^ 1);
    }
    buf ^= 1;
    if (__syncthreads_and(wave_done)) break;
  }
  if (a.tile_work && v == 0 && tid == 0) a.tile_work[tile] = make_uint2(range.y - range.x, consumed);
  if (inside) a.pixels[v][(size_t)py * W + px] = pix.packed(a.bgra != 0);
}

void launch_bin(const BinLaunch& a, hipStream_t s) {
  const dim3 grid(a.grid_x, a.views), block(kBinThreads);
  if (a.items == 1) hipLaunchKernelGGL((k_bin<kBinThreads, 1>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_bin<kBinThreads, kBinItems>), grid, block, 0, s, a);
}

void launch_ranges(const RangesLaunch& a, hipStream_t s) {
  hipLaunchKernelGGL(k_tile_ranges, dim3(a.grid_x, a.views), dim3(256), 0, s, a);
}

template <bool UNALIGNED, bool F32, int MODE>
void launch_raster_as(bool small, dim3 grid, dim3 block, hipStream_t s, const RasterLaunch& a) {
  if (small) hipLaunchKernelGGL((k_raster<UNALIGNED, F32, MODE, 128>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_raster<UNALIGNED, F32, MODE, 256>), grid, block, 0, s, a);
}

template <bool UNALIGNED, bool F32>
void launch_raster_mode(bool small, dim3 grid, dim3 block, hipStream_t s, const RasterLaunch& a) {
  if (a.walk == 3) launch_raster_as<UNALIGNED, F32, 3>(small, grid, block, s, a);
  else if (a.walk == 2) launch_raster_as<UNALIGNED, F32, 2>(small, grid, block, s, a);
  else if (a.walk == 1) launch_raster_as<UNALIGNED, F32, 1>(small, grid, block, s, a);
  else launch_raster_as<UNALIGNED, F32, 0>(small, grid, block, s, a);
}

void launch_raster(const RasterLaunch& a, hipStream_t s) {
  const dim3 grid(a.grid_x), block(256);
  const bool small = a.batch_entries == 128;
  if (a.use_unaligned_rectangles) {
    if (a.blend_f32) launch_raster_mode<true, true>(small, grid, block, s, a);
    else launch_raster_mode<true, false>(small, grid, block, s, a);
  } else {
    if (a.blend_f32) launch_raster_mode<false, true>(small, grid, block, s, a);
    else launch_raster_mode<false, false>(small, grid, block, s, a);
  }
}

}  // namespace spl
