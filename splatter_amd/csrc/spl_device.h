// spl_device.h -- device helpers shared by the splat pipeline kernels
// (gfx950: wave64, 160 KB LDS per CU, 8 XCDs with private L2s).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "spl_internal.h"

namespace spl {

constexpr int kWave = 64;

// Lookback status words: 2 flag bits + 30-bit count (shaders.wgsl:438-457
// uses the same split: 0x4... aggregate, 0x8... inclusive prefix).
constexpr uint32_t kFlagAggregate = 0x40000000u;
constexpr uint32_t kFlagInclusive = 0x80000000u;
constexpr uint32_t kFlagMask = 0xC0000000u;
constexpr uint32_t kCountMask = 0x3FFFFFFFu;

// Number of set bits of `mask` held by lanes below this one.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint32_t lane_id() { return lanes_below(~0ull); }

// Status words are read and written at agent scope so that the per-XCD L2s
// do not hide one tile's publication from a tile running on another XCD.
__device__ __forceinline__ uint32_t load_status(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_status(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Look-back for one digit counter that inspects WIN predecessors per step
// (their loads are issued together), so the wait for an inclusive prefix
// that is t tiles away costs t/WIN memory round trips instead of t.
// Publishes nothing: the caller publishes the aggregate beforehand and the
// inclusive prefix (returned + count) afterwards.
template <int WIN>
__device__ __forceinline__ uint32_t lookback_window(const uint32_t* status, uint32_t tile, size_t stride) {
  static_assert(WIN <= 32, "window masks are 32 bits");
  uint32_t prefix = 0;
  int64_t p = (int64_t)tile - 1;
  while (true) {
    uint32_t s[WIN];
    uint32_t inv = 0, inc = 0;
#pragma unroll
    for (int i = 0; i < WIN; ++i) {
      s[i] = (p - i >= 0) ? load_status(status + (size_t)(p - i) * stride) : kFlagInclusive;
      inv |= ((s[i] & kFlagMask) == 0 ? 1u : 0u) << i;
      inc |= ((s[i] & kFlagInclusive) != 0 ? 1u : 0u) << i;
    }
    const uint32_t first_inv = inv ? (uint32_t)__builtin_ctz(inv) : (uint32_t)WIN;
    const uint32_t first_inc = inc ? (uint32_t)__builtin_ctz(inc) : (uint32_t)WIN;
    const bool done = first_inc < first_inv;
    const uint32_t take = done ? first_inc + 1 : first_inv;  // words summed this round
#pragma unroll
    for (int i = 0; i < WIN; ++i) prefix += (uint32_t)i < take ? (s[i] & kCountMask) : 0u;
    if (done) break;
    p -= take;
    if (take < (uint32_t)WIN) __builtin_amdgcn_s_sleep(1);
  }
  return prefix;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__device__ __forceinline__ uint64_t wave_sum64(uint64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

// Look-back for a single counter per tile run by one whole wave: the 64
// lanes read the 64 nearest predecessors at once and a ballot finds the
// nearest inclusive prefix (or the first not yet published).  Returns the
// exclusive prefix in every lane; lane 0 publishes aggregate and inclusive.
__device__ __forceinline__ uint32_t wave_lookback(uint32_t* status, uint32_t tile, uint32_t count) {
  const uint32_t lane = lane_id();
  if (tile == 0) {
    if (lane == 0) store_status(status, kFlagInclusive | count);
    return 0;
  }
  if (lane == 0) store_status(status + tile, kFlagAggregate | count);
  uint32_t prefix = 0;
  int64_t base = (int64_t)tile - 1;
  while (true) {
    const int64_t i = base - (int64_t)lane;
    const uint32_t s = i >= 0 ? load_status(status + i) : kFlagInclusive;
    const uint64_t inv = __ballot((s & kFlagMask) == 0);
    const uint64_t inc = __ballot((s & kFlagInclusive) != 0);
    const uint32_t first_inc = inc ? (uint32_t)__builtin_ctzll(inc) : 64u;
    const uint32_t first_inv = inv ? (uint32_t)__builtin_ctzll(inv) : 64u;
    if (first_inc < first_inv) {
      prefix += wave_sum(lane <= first_inc ? (s & kCountMask) : 0u);
      break;
    }
    prefix += wave_sum(lane < first_inv ? (s & kCountMask) : 0u);
    base -= first_inv;
    if (first_inv < 64u) __builtin_amdgcn_s_sleep(1);
  }
  if (lane == 0) store_status(status + tile, kFlagInclusive | (prefix + count));
  return prefix;
}

// 64-bit variant for counts that may pass 2^30 (screen-tile pairs): flags in
// the top two bits, 62-bit count.
constexpr uint64_t kFlagAggregate64 = 1ull << 62;
constexpr uint64_t kFlagInclusive64 = 1ull << 63;
constexpr uint64_t kCountMask64 = (1ull << 62) - 1;

__device__ __forceinline__ uint64_t wave_lookback64(uint64_t* status, uint32_t tile, uint64_t count) {
  const uint32_t lane = lane_id();
  auto ld = [](const uint64_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto st = [](uint64_t* p, uint64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  if (tile == 0) {
    if (lane == 0) st(status, kFlagInclusive64 | count);
    return 0;
  }
  if (lane == 0) st(status + tile, kFlagAggregate64 | count);
  uint64_t prefix = 0;
  int64_t base = (int64_t)tile - 1;
  while (true) {
    const int64_t i = base - (int64_t)lane;
    const uint64_t s = i >= 0 ? ld(status + i) : kFlagInclusive64;
    const uint64_t inv = __ballot((s >> 62) == 0);
    const uint64_t inc = __ballot((s & kFlagInclusive64) != 0);
    const uint32_t first_inc = inc ? (uint32_t)__builtin_ctzll(inc) : 64u;
    const uint32_t first_inv = inv ? (uint32_t)__builtin_ctzll(inv) : 64u;
    if (first_inc < first_inv) {
      prefix += wave_sum64(lane <= first_inc ? (s & kCountMask64) : 0ull);
      break;
    }
    prefix += wave_sum64(lane < first_inv ? (s & kCountMask64) : 0ull);
    base -= first_inv;
    if (first_inv < 64u) __builtin_amdgcn_s_sleep(1);
  }
  if (lane == 0) st(status + tile, kFlagInclusive64 | (prefix + count));
  return prefix;
}

// Exclusive scan of one value per thread over a block of THREADS threads.
// s_tmp holds THREADS/64 words.  Contains two barriers.
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_tmp, uint32_t& total) {
  constexpr int WAVES = THREADS / kWave;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  // Blocks of sixteen waves tell the compiler that the wave index is uniform:
  // otherwise its address in s_tmp and the sixteen comparisons below stay in
  // registers across a caller's loop, and a radix-sort pass of 16 keys a lane
  // reloaded that address from scratch in every tile, behind a wait for its
  // value loads (1.5M pairs by count 41.6 us, 40.7 so; 11.8M 117 and 115).  Smaller
  // blocks have the registers (depth sort of 1M splats, 512 x 8: 57.7 us, 58.5
  // with the uniform index).
  uint32_t w = threadIdx.x / kWave;
  if constexpr (WAVES > 8) w = __builtin_amdgcn_readfirstlane(w);
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    uint32_t y = __shfl_up(x, o, kWave);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == kWave - 1) s_tmp[w] = x;
  __syncthreads();
  uint32_t before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    uint32_t t = s_tmp[i];
    before += (i < (int)w) ? t : 0u;
    tot += t;
  }
  total = tot;
  __syncthreads();
  return before + x - v;
}

// Tickets of a persistent grid.  Blocks take tiles in order from a counter:
// an atomic on one address costs about 11.5 ns however many blocks issue it
// (1024 tickets 11.8 us, measured), so a launch spends as few as it can.
// Blocks past the number of tiles leave without a ticket.  Where every tile
// has a block, each of those draws one and is done (a second ticket would cost
// a block another microsecond to learn that there are no more); otherwise
// every block's last ticket is past the tiles.  Either way the number of
// tickets is known, and whoever draws the last one resets the counter for the
// next launch.  No second counter and no fence: the tickets before the last
// have been drawn, and the launch's end publishes the reset.  (A counter of
// leaving blocks behind a __threadfence, which writes an XCD's L2 back, cost
// 1024 blocks 20 to 40 us.)
__device__ __forceinline__ bool persistent_idle(uint32_t num_tiles) { return blockIdx.x >= num_tiles; }
__device__ __forceinline__ bool one_tile_each(uint32_t num_tiles) { return gridDim.x >= num_tiles; }

__device__ __forceinline__ uint32_t take_ticket(uint32_t* counter, uint32_t num_tiles) {
  const uint32_t t = atomicAdd(counter, 1u);
  const uint32_t tickets = one_tile_each(num_tiles) ? num_tiles : num_tiles + gridDim.x;
  if (t == tickets - 1u) atomicExch(counter, 0u);
  return t;
}

// The tile of a pass over `count` keys that goes by their number: the smaller
// while one round of blocks (one of 1024 lanes a CU, `one_round` keys) holds
// them all.
__device__ __forceinline__ uint32_t by_count_tile(uint32_t count, uint32_t one_round) {
  return count <= one_round ? kTileNarrow : kTileWide;
}

// Words of a finished sort pass's status to zero: of the capacity's `words`,
// those of the tiles (`tile` keys, at most 256 digits) that `count` keys had;
// tile 0: all.
__device__ __forceinline__ size_t used_status(size_t words, uint32_t tile, uint32_t one_round, uint32_t count) {
  if (tile == kTileByCount) tile = by_count_tile(count, one_round);
  const size_t used = tile ? ((size_t)count + tile - 1) / tile * 256 : words;
  return used < words ? used : words;
}

// Grid-stride zeroing of another stage's finished bookkeeping.
__device__ __forceinline__ void clear_words(uint32_t* p, size_t n) {
  if (!p) return;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0u;
}

}  // namespace spl
