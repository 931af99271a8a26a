// A scatter by digit whose order within a digit's run is free: the MSD
// sort's scatter by the top 10-bit digit (k_msd.hip) and the learned sort's
// two scatters by bucket (k_learned.hip), whose buckets are all sorted
// afterwards. Shared by both.
//
// Such a scatter needs no lookback. A tile (one workgroup) counts its keys
// per digit with LDS atomics, whose returned value is the key's rank in the
// tile's run of that digit; one thread per digit then claims the run's place
// in the segment with one atomic add on the digit's cursor (zeroed before
// the launch), on top of the digit's start in the segment, an exclusive scan
// of the segment's digit counts. Keys are staged in LDS in digit order and
// written with consecutive threads on consecutive slots of each run.
//
// A tile is a chain of load, count, claim, place and store with a barrier
// between each, so what counts is how many tiles share a CU: with at most 64
// registers (ranks two a register, cheap digits recomputed, rows at scalar
// addresses, one path for whole and partial tiles) two of 16 waves do instead of
// one. The MSD scatter of 10M keys 41 -> 36 us, of 2^24 clustered ones 51 -> 42.
#pragma once

#include <type_traits>

#include "ocp_internal.hpp"

namespace ocp {

// The top 10-bit digit of a 30-bit key.
struct TopDigit10 {
  static constexpr bool kCheap = true;
  static constexpr int kBits = 10;
  __device__ __forceinline__ void setup(int32_t, int, int) const {}
  __device__ __forceinline__ uint32_t operator()(uint32_t key) const {
    return (key >> 20) & 1023u;
  }
};

// A tile's work, one workgroup: the keys in[base, base + cnt) of a segment
// [sb, sb + len). Digit functor: kBits, kCheap (recomputed from the key rather
// than staged in LDS) and the digit of a key. hist[d]: the segment's count of
// digit d; cursor[d]: its zeroed claim counters. extra(digits, keys) runs once
// the keys are in registers, before they are placed.
template <int THREADS, int KPT, class Digit, class Extra>
__device__ __forceinline__ void cursor_scatter_tile(
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int32_t sb, int32_t len,
    int32_t base, int32_t cnt, const uint32_t* __restrict__ hist, uint32_t* __restrict__ cursor,
    Digit dig, Extra extra) {
  constexpr int RADIX = 1 << Digit::kBits;
  constexpr int T = THREADS * KPT;
  constexpr bool CHEAP = Digit::kCheap;
  static_assert(THREADS >= RADIX, "one thread per digit");
  using DigT = typename std::conditional<(RADIX > 256), uint16_t, uint8_t>::type;
  __shared__ uint32_t s_keys[T];
  __shared__ DigT s_dig[CHEAP ? 1 : T];
  __shared__ uint32_t s_run[RADIX + 64];  // tile counts, then the LDS start of each run
  __shared__ int32_t s_gpos[RADIX];  // global slot of a run's LDS slot 0
  __shared__ uint32_t s_tmp[2 * (THREADS / 64)];
  const int tid = threadIdx.x;
  if (tid < RADIX) s_run[tid] = 0;
  if (tid < 64) s_run[RADIX + tid] = 0;
  const uint32_t hv = tid < RADIX ? hist[tid] : 0u;
  uint32_t keys[KPT];
  // (rows at scalar addresses: one register of offsets for all of them)
  const uint32_t* src = in + __builtin_amdgcn_readfirstlane(base);
  if (cnt == T) {
#pragma unroll
    for (int k = 0; k < KPT; ++k) keys[k] = (src + k * THREADS)[tid];
  } else {
#pragma unroll
    for (int k = 0; k < KPT; ++k) keys[k] = src[min(k * THREADS + tid, cnt - 1)];
  }
  __syncthreads();
  // Past the tile's keys: digits of their own, one a lane, so that one code
  // without branches serves whole and partial tiles; what they place lies past
  // the tile's last slot (and need not be one slot each).
  const auto digit = [&](int k) {
    return k * THREADS + tid < cnt ? dig(keys[k]) : RADIX + (tid & 63u);
  };
  uint32_t dg[KPT], rank[(KPT + 1) / 2];  // ranks are below 2^16, two a register
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    dg[k] = digit(k);
    const uint32_t r = atomicAdd(&s_run[dg[k]], 1u);
    if (k & 1) rank[k / 2] |= r << 16;
    else rank[k / 2] = r;
  }
  __syncthreads();
  extra(hv, dg, keys);
  const uint32_t c = tid < RADIX ? s_run[tid] : 0u;
  uint32_t lstart, gbase;
  block_excl_scan2<THREADS>(c, hv, s_tmp, &lstart, &gbase);
  if (tid < RADIX) {
    int32_t gpos = 0;
    if (c)
      gpos = sb + static_cast<int32_t>(gbase + atomicAdd(&cursor[tid], c)) -
             static_cast<int32_t>(lstart);
    s_run[tid] = lstart;  // (every read of the counts came before the scan's barriers)
    s_gpos[tid] = gpos;
  }
  if (tid < 64) s_run[RADIX + tid] = static_cast<uint32_t>(cnt);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const uint32_t d = CHEAP ? digit(k) : dg[k];  // (a cheap one is not held across the barriers)
    const uint32_t pos = s_run[d] + ((rank[k / 2] >> ((k & 1) * 16)) & 0xffffu);
    s_keys[pos] = keys[k];
    if constexpr (!CHEAP) s_dig[pos] = static_cast<DigT>(d);
  }
  __syncthreads();
  // The LDS reads of a batch in flight together, then its stores.
  constexpr int BATCH = KPT % 4 == 0 ? 4 : 1;
#pragma unroll 1
  for (int32_t i0 = tid; i0 < cnt; i0 += BATCH * THREADS) {
    uint32_t key[BATCH];
    int32_t to[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      key[k] = s_keys[i0 + k * THREADS];  // (a batch ends at or before T)
      if constexpr (!CHEAP) to[k] = s_dig[i0 + k * THREADS];
    }
#pragma unroll
    for (int k = 0; k < BATCH; ++k)
      to[k] = s_gpos[(CHEAP ? dig(key[k]) : static_cast<uint32_t>(to[k])) & (RADIX - 1u)] + i0 +
              k * THREADS;
    // (inside the segment whenever the counts describe these keys, as the
    // launchers' counts do)
#pragma unroll
    for (int k = 0; k < BATCH; ++k)
      if (i0 + k * THREADS < cnt &&
          static_cast<uint32_t>(to[k] - sb) < static_cast<uint32_t>(len))
        out[to[k]] = key[k];
  }
}

struct NoExtra {
  template <int KPT>
  __device__ __forceinline__ void operator()(uint32_t, const uint32_t (&)[KPT],
                                             const uint32_t (&)[KPT]) const {}
};

// One tile per workgroup, tiles of THREADS * KPT keys that never straddle a
// segment. The functor's setup(seg, tid, threads) fills per-segment LDS
// tables. hist[seg * hstride + d], cursor[seg * 2^kBits + d]; tiles_dev
// (optional): the number of real tiles when the grid is sized for an upper
// bound.
template <int THREADS, int KPT, class Digit>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(8))) void cursor_scatter_kernel(
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out, SegView sv,
    const int32_t* __restrict__ tile_start, const int32_t* __restrict__ tiles_dev,
    const uint32_t* __restrict__ hist, int64_t hstride, uint32_t* __restrict__ cursor,
    const uint32_t* __restrict__ ctrl, Digit dig) {
  constexpr int RADIX = 1 << Digit::kBits;
  constexpr int T = THREADS * KPT;
  const int32_t t = static_cast<int32_t>(blockIdx.x);
  if (tiles_dev && t >= *tiles_dev) return;
  if (stopped_any(ctrl)) return;
  const TileRef r = find_tile(tile_start, sv.n_seg, t);
  const int32_t sb = seg_begin(sv, r.seg);
  const int32_t len = seg_end(sv, r.seg) - sb;
  const int32_t base = sb + r.local * T;
  dig.setup(r.seg, threadIdx.x, THREADS);
  cursor_scatter_tile<THREADS, KPT>(in, out, sb, len, base, min(T, sb + len - base),
                                    hist + static_cast<int64_t>(r.seg) * hstride,
                                    cursor + static_cast<int64_t>(r.seg) * RADIX, dig, NoExtra{});
}

}  // namespace ocp
