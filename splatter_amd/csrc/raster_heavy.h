// raster_heavy.h -- the rasteriser of the tiles with the longest lists
// (k_heavy_tiles), part of k_raster.
//
// A tile's entries blend one after another, so a list of tens of thousands
// sets the frame's time however idle the rest of the chip is: what bounds it
// is the latency of each round of gather, test and blend.  Such a tile takes
// eight blocks, one per 8x4 pixels, of two producer and two consumer waves.
// The producers gather the list 128 entries at a time, only the row with the
// pixel box at first, then the other two rows of the entries whose box meets
// the block's pixels, and append those, prepared, to a ring in LDS, in order.
// Each consumer owns a 4x4 sub-block and takes the ring 64 entries at a time:
// it first finds, entry-parallel (one lane per entry, sixteen exact per-pixel
// tests), the 64-bit mask of the entries that cover each pixel; then four
// lanes per pixel evaluate its next four covering entries side by side, and
// blend them in order with one colour channel (or the transmittance) per
// lane.  The arithmetic per fragment and its order are the other walks', so
// the pixels are the same.
//
// Raster of one 640x480 view of 1.5M splats (longest list 27021): 302 us with
// four blocks of the ordinary walk on such a tile, 160 so; 400k splats with
// squares and the f32 blend 227 against 94 us.  Also measured there: sixteen
// blocks of 4x4 with three producers gathering whole records 257 us (the
// gathers fill the L1s), 199 with a tile's blocks on one XCD.
#pragma once
#include "raster_common.h"

namespace spl {

namespace {

constexpr uint32_t kBatch = 128;  // entries the producers stage per round
constexpr uint32_t kRing = 256;   // entries; an append that does not fit waits a round (63 at most are left then)

// The compiler's v_writelane_b32 (value and lane uniform), which has no
// builtin of its own: lane `at` of the result is `value`, the others are `old`.
// A compiler without the intrinsic of this name refuses the file; the plain
// form, lane == at ? value : old, takes two instructions and spills registers of
// the ordinary tiles' walk beside it (raster of 6M splats at 1080p 321 us so,
// 335 with it; 400k with the f32 blend 100 and 104).
__device__ uint32_t writelane(uint32_t value, uint32_t at, uint32_t old) __asm("llvm.amdgcn.writelane.i32");

// quad_perm broadcasts and swaps (DPP)
template <int CTRL>
__device__ __forceinline__ float quad(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
// A copy in a register that holds nothing else.
template <typename T>
__device__ __forceinline__ void own(T& to, T from) {
  asm volatile("v_mov_b32 %0, %1" : "=&v"(to) : "v"(from));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kQuadLast = 0xFF;

// One block's share of a heavy tile: the 8x4 pixels number `part` of it.
// ring: 3 x kRing entries' rows; words: 8 words of LDS.
template <bool UNALIGNED, bool F32>
__device__ __forceinline__ void raster_heavy(const RasterLaunch& a, uint32_t v, uint32_t tile, uint32_t part,
                                             float4* ring, uint32_t* words) {
  float4 *const s_m = ring, *const s_t = ring + kRing, *const s_c = ring + 2 * kRing;
  // by round parity: entries each producer wave kept of its batch, and whether
  // each sub-block still takes fragments
  uint4* const s_round = reinterpret_cast<uint4*>(words);
  const Uniforms& u = a.uniforms[v];
  const uint32_t* pair_vals = a.pair_vals + v * a.pair_stride;
  const float4* records = a.records + v * a.rec_stride;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  const bool producer = w < 2u;
  const uint32_t W = u.image_size[0], H = u.image_size[1];
  const uint32_t qx0 = (tile % u.tiles_x) * kTileSize + (part & 1u) * 8u;
  const uint32_t qy0 = (tile / u.tiles_x) * kTileSize + (part >> 1) * 4u;
  if (qx0 >= W || qy0 >= H) return;
  uint2 range = a.ranges[v * a.ranges_stride + tile];
  range.x &= ~kHeavyFlag;
  const PixelMap pm = pixel_map(u);
  const float margin = u.ellipse_margin;
  const uint32_t visible = a.counters[(size_t)v * kCounterWords + kVisible];

  // consumer: lane 4p + ch holds channel ch (r, g, b, transmittance) of pixel p of its sub-block
  const uint32_t ch = lane & 3u, p = lane >> 2;
  const uint32_t bx0 = qx0 + (w & 1u) * 4u, by0 = qy0;
  const uint32_t px = bx0 + (p & 3u), py = by0 + (p >> 2);
  const float pxf = (float)px, pyf = (float)py;
  const bool inside = px < W && py < H;
  const bool odd = (ch & 1u) != 0u, upper = (ch & 2u) != 0u;
  float x = ch == 3u ? (F32 ? 1.0f : 255.0f) : 0.0f;

  // producer: record index and box row of this lane's entry in the batch to
  // stage, the index after that, and the rows of the entry it kept last
  uint32_t c0 = 0, i1 = 0;
  float4 g0 = make_float4(0, 0, 0, 0), g1 = g0, g2 = g0;
  float tx = 0.0f, ty = 0.0f;
  bool keep = false;
  const auto index_at = [&](uint32_t base) -> uint32_t {
    const uint32_t i = base + tid;
    return pair_vals[i < range.y ? i : range.x];
  };
  // (an index past the records, only after an upstream error, reads record 0)
  const auto row = [&](uint32_t c, uint32_t k) { return records[3 * (size_t)(c < visible ? c : 0u) + k]; };
  if (producer) {
    c0 = index_at(range.x);
    i1 = index_at(range.x + kBatch);
    g2 = row(c0, 2);
  }

  uint32_t head = 0, tail = 0;   // entries appended and taken
  uint32_t pend = 0, before = 0; // entries kept by the last staged batch, not appended yet; of those, by lower waves
  uint32_t base = range.x;       // the batch the producers stage next
  uint32_t par = 0;
  bool live0 = true, live1 = true;  // sub-blocks that still take fragments
  __syncthreads();
  while (true) {
    const uint32_t ready = head - tail;
    const bool fits = ready + pend <= kRing;
    const bool last = base >= range.y && pend == 0u;
    const uint32_t take = last ? ready : ready & ~63u;
    const bool staging = fits && base < range.y;
    if (producer) {
      float4 e0, e1, e2;
      prepare_entry<UNALIGNED>(g0, g1, make_float4(tx, ty, 0.0f, 0.0f), pm, margin, e0, e1, e2);
      const uint64_t kept = __ballot(keep);
      const uint32_t at = (head + before + lanes_below(kept)) & (kRing - 1u);
      const bool append = fits && keep;
      if (append) {
        s_m[at] = e0;
        s_t[at] = e1;
        s_c[at] = e2;
      }
      if (fits) keep = false;
      if (staging) {
        const uint32_t lo = __float_as_uint(g2.z), hi = __float_as_uint(g2.w);
        const uint32_t x0 = qx0 + (live0 ? 0u : 4u), x1 = qx0 + (live1 ? 7u : 3u);
        keep = base + tid < range.y && lo != 0xFFFFFFFFu && (lo & 0xFFFFu) <= x1 && (hi & 0xFFFFu) >= x0 &&
               (lo >> 16) <= qy0 + 3u && (hi >> 16) >= qy0;
        const uint64_t bm = __ballot(keep);
        if (lane == 0) words[4u * par + w] = (uint32_t)__popcll(bm);
        own(tx, g2.x);
        own(ty, g2.y);
        const uint32_t ck = keep ? c0 : 0u;  // (entries not kept read record 0, one line)
        __builtin_amdgcn_sched_barrier(0);
        g0 = row(ck, 0);
        g1 = row(ck, 1);
        own(c0, i1);
        g2 = row(c0, 2);
        i1 = index_at(base + 2u * kBatch);
      }
    } else {
      for (uint32_t done = 0; done < take; done += 64u) {
        const uint32_t first = tail + done;
        const uint32_t cnt = min(64u, take - done);
        uint32_t lo, hi;
        {
          // lane = entry: the exact test at each of the sub-block's pixels
          const uint32_t k = (first + lane) & (kRing - 1u);
          const float4 m = s_m[k];
          float4 t = s_t[k];
          t.z = lane < cnt ? (UNALIGNED ? margin * kGaussScale : t.z) : -1.0f;  // covers nothing
          uint32_t vlo = 0, vhi = 0;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            float uu, ww;
            const bool c = covers<UNALIGNED>(m, t, (float)(bx0 + (i & 3)), (float)(by0 + (i >> 2)), pm, uu, ww);
            const uint64_t bal = __ballot(c);
            vlo = writelane((uint32_t)bal, i, vlo);
            vhi = writelane((uint32_t)(bal >> 32), i, vhi);
          }
          lo = (uint32_t)__shfl((int)vlo, (int)p, kWave);
          hi = (uint32_t)__shfl((int)vhi, (int)p, kWave);
        }
        if (quad<kQuadLast>(x) == 0.0f || !inside) lo = hi = 0u;
        uint32_t off = 0;
        if (lo == 0u) { lo = hi; hi = 0u; off = 32u; }
        while (__ballot(lo != 0u)) {
          // this pixel's next four entries, one per lane
          const uint32_t m1 = lo & (lo - 1u), m2 = m1 & (m1 - 1u), m3 = m2 & (m2 - 1u);
          const uint32_t low = odd ? m1 : lo, high = odd ? m3 : m2;
          const uint32_t mine = upper ? high : low;
          const bool has = mine != 0u;
          const uint32_t k = (first + off + (uint32_t)__builtin_ctz(mine | 0x80000000u)) & (kRing - 1u);
          const float4 m = s_m[k], t = s_t[k], col = s_c[k];
          float uu, ww;
          (void)covers<UNALIGNED>(m, t, pxf, pyf, pm, uu, ww);
          const float alpha = t.w * spl_exp2(-fmaf(uu, uu, ww * ww));
          const bool ok = has && alpha >= 1.0f / 255.0f;
          const float al = ok ? alpha : 0.0f;
          float f0, f1, f2;
          const float f3 = -al;
          if constexpr (F32) {
            f0 = ok ? col.x * al : 0.0f;
            f1 = ok ? col.y * al : 0.0f;
            f2 = ok ? col.z * al : 0.0f;
          } else {
            f0 = clamp01(col.x * al);
            f1 = clamp01(col.y * al);
            f2 = clamp01(col.z * al);
          }
          // transpose within the quad: s[j] = entry j's factor for this
          // channel (every swap runs in all lanes, then each lane selects)
          const float d0 = quad<kQuadXor1>(f0), d1 = quad<kQuadXor1>(f1);
          const float d2 = quad<kQuadXor1>(f2), d3 = quad<kQuadXor1>(f3);
          const float a0 = odd ? d1 : f0, a1 = odd ? f1 : d0, a2 = odd ? d3 : f2, a3 = odd ? f3 : d2;
          const float b0 = quad<kQuadXor2>(a0), b1 = quad<kQuadXor2>(a1);
          const float b2 = quad<kQuadXor2>(a2), b3 = quad<kQuadXor2>(a3);
          const float s[4] = {upper ? b2 : a0, upper ? b3 : a1, upper ? a2 : b0, upper ? a3 : b1};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float tr = quad<kQuadLast>(x);
            const float y = fmaf(s[j], tr, x);
            if constexpr (F32) x = tr == 0.0f ? x : y;
            else x = fminf(rintf(y), 255.0f);
          }
          lo = m3 & (m3 - 1u);
          if (lo == 0u) { lo = hi; hi = 0u; off = 32u; }
          if (quad<kQuadLast>(x) == 0.0f) lo = hi = 0u;
        }
      }
      const uint64_t live = __ballot(ch == 3u && inside && x != 0.0f);
      if (lane == 0) words[4u * par + w] = live ? 1u : 0u;
    }
    __syncthreads();
    const uint4 round = s_round[par];
    if (fits) { head += pend; pend = 0u; }
    tail += take;
    if (staging) {
      pend = round.x + round.y;
      before = w == 1u ? round.x : 0u;
      base += kBatch;
    }
    live0 = round.z != 0u;
    live1 = round.w != 0u;
    if (!(live0 || live1) || (last && tail == head)) break;
    par ^= 1u;
  }
  if (a.tile_work && v == 0 && tid == 0)
    atomicMax(&a.tile_work[tile].y, min(base, range.y) - range.x);
  if (!producer) {
    uint32_t code = F32 ? (uint32_t)q8(x) : (uint32_t)x;
    const uint32_t pos = ch == 3u || !a.bgra ? ch : 2u - ch;
    code <<= 8u * pos;
    code |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)code, kQuadXor1, 0xF, 0xF, true);
    code |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)code, kQuadXor2, 0xF, 0xF, true);
    if (inside && ch == 0u) a.pixels[v][(size_t)py * W + px] = code;
  }
}

}  // namespace

}  // namespace spl
