// LDS radix sort of one bucket of 32-bit keys by one workgroup, shared by
// the learned-CDF bucket sort (k_learned.hip) and the MSD sort of a build's
// keys (k_msd.hip).
#pragma once

#include "ocp_internal.hpp"

namespace ocp {

// Sorts src[0, n) into g[0, n) (which may be the same), 0 < n <= WAVES * 64 *
// KPT: keys are loaded wave-contiguously, taken relative to the bucket
// minimum, and sorted by LSD passes over the bits they span - a counting sort
// with LDS atomics over the low P0 bits (one counter per digit), then stable
// passes of up to P1 bits ranked per wave by ballot multisplit - scattered
// through LDS. Every thread of the workgroup calls it, any number of times.
// With span > 0 the caller knows every key lies in [base, base + 2^span)
// and the workgroup skips finding the bucket's range.
//
// With BINS the keys are first counted into 2^BINS equal parts of the span by
// LDS atomics, whose returned value places a key in its part; where no part
// holds kBinMax keys, a key's rank among its part's few, found by comparing
// them, is its final place, and the two radix passes are not needed. That is
// how spread keys are sorted (10M uniform points in digits of 9,800 keys: 58 ->
// 47 us); keys that crowd into few parts take the radix passes. More than 16
// in a part (32, 64) cost clustered clouds 30-130% of their windows' time.
constexpr uint32_t kBinMax = 16;

// Adds `unit` to a digit's counter in LDS and returns what it was. Adds of one wave
// to one counter are made one after the other; with SHARED the lanes that have the
// first lane's digit are added at once, where there are several.
template <bool SHARED>
__device__ __forceinline__ uint32_t count_digit(uint32_t* counter, uint32_t digit, uint32_t unit) {
  if constexpr (SHARED) {
    const uint32_t first = static_cast<uint32_t>(
        __builtin_amdgcn_readfirstlane(static_cast<int>(digit)));
    const uint64_t same = __ballot(digit == first);
    const uint32_t n = static_cast<uint32_t>(__popcll(same));
    if (n >= 8u && digit == first) {
      const uint32_t rank = static_cast<uint32_t>(__popcll(same & lanemask_lt()));
      uint32_t old = 0;
      if (rank == 0) old = atomicAdd(counter, n * unit);
      old = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(old)));
      return old + rank * unit;
    }
  }
  return atomicAdd(counter, unit);
}

// SHARED (see count_digit): for keys of which many may be equal, or equal in the
// bits that a pass looks at.
template <int WAVES, int KPT, int P0 = (WAVES >= 16 ? 12 : WAVES == 8 ? 11 : 10), int P1 = 8,
          int BINS = 0, bool SHARED = false>
__device__ __forceinline__ void lds_bucket_sort(const uint32_t* src, uint32_t* g, int32_t n,
                                                uint32_t base = 0, int span = 0) {
  constexpr int THREADS = WAVES * 64;
  constexpr int CAP = THREADS * KPT;
  // First-pass counters (2^P0) and the stable passes' per-wave digit
  // counters share one array.
  constexpr int NB = 1 << P0;
  constexpr int ND = 1 << P1;
  constexpr int HW = NB > WAVES * ND ? NB : WAVES * ND;
  // Digits per thread when the stable passes' counters are scanned.
  constexpr int DPT = ND > THREADS ? ND / THREADS : 1;
  static_assert(P0 >= 8 && NB % THREADS == 0, "whole counters per thread");
  __shared__ uint32_t s_keys[CAP];
  __shared__ uint32_t s_whist[HW];
  __shared__ uint32_t s_dstart[ND];
  __shared__ uint32_t s_tmp[WAVES];
  __shared__ uint32_t s_mm[2];
  const int tid = threadIdx.x;
  const uint32_t w = wave_id();
  // (opaque, so that a caller's loop does not keep every row's addresses)
  uint32_t lane = lane_id();
  asm volatile("" : "+v"(lane));
  if (tid == 0) {
    s_mm[0] = 0xffffffffu;
    s_mm[1] = 0u;
  }
  // Each wave owns `rows` rows of 64 consecutive keys, as few as hold n keys, so
  // that every wave has its share; a row that starts at or past n holds padding
  // only and is left out of every pass.
  const int rows = (n + THREADS - 1) / THREADS;
  const int32_t wbase = static_cast<int32_t>(w) * (64 * rows);
  const int32_t wend = min(n, wbase + 64 * rows);
  uint32_t kv[KPT];
  uint32_t mn = 0xffffffffu, mx = 0u;
  // All loads first (consuming each in its own iteration keeps one load in
  // flight per wave), then the bucket's range.
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
    kv[k] = idx < wend ? src[idx] : 0u;
  }
  int bits = span;
  if (span > 0) {
    mn = base;
  } else {
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
      if (idx < wend) {
        mn = min(mn, kv[k]);
        mx = max(mx, kv[k]);
      }
    }
    mn = wave_min(mn);
    mx = wave_max(mx);
    __syncthreads();
    if (lane == 0) {
      atomicMin(&s_mm[0], mn);
      atomicMax(&s_mm[1], mx);
    }
    __syncthreads();
    mn = s_mm[0];
    mx = s_mm[1];
    if (mn == mx) return;  // constant bucket: already sorted
    bits = 32 - __clz(static_cast<int>(mx - mn));
  }
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
    kv[k] = idx < wend ? kv[k] - mn : 0xffffffffu;  // padding ranks last
  }
  if constexpr (BINS > 0) {
    // Two 16-bit counters a word, then the parts' starts.
    constexpr int NP = 1 << BINS;
    constexpr int WPT = NP / 2 / THREADS;  // words per thread
    static_assert(CAP < 65536 && NP / 2 <= HW && WPT * THREADS * 2 == NP, "parts fit");
    const int low = bits > BINS ? bits - BINS : 0;
    for (int i = tid; i < NP / 2; i += THREADS) s_whist[i] = 0;
    __syncthreads();
    uint32_t at[KPT];
    bool crowded = false;
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      if (wbase + k * 64 >= wend) continue;
      const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
      if (idx < wend) {
        const uint32_t b = kv[k] >> low, sh = (b & 1u) * 16u;
        at[k] = (count_digit<SHARED>(&s_whist[b >> 1], b, 1u << sh) >> sh) & 0xffffu;
        crowded |= at[k] >= kBinMax;
      }
    }
    if (!__syncthreads_or(crowded)) {
      uint32_t cc[WPT];
      uint32_t sum = 0;
#pragma unroll
      for (int j = 0; j < WPT; ++j) {
        cc[j] = s_whist[tid * WPT + j];
        sum += (cc[j] & 0xffffu) + (cc[j] >> 16);
      }
      uint32_t all;
      uint32_t run = block_excl_scan<THREADS>(sum, s_tmp, &all);
#pragma unroll
      for (int j = 0; j < WPT; ++j) {
        const uint32_t mid = run + (cc[j] & 0xffffu);
        s_whist[tid * WPT + j] = run | (mid << 16);
        run = mid + (cc[j] >> 16);
      }
      __syncthreads();
      const uint16_t* start = reinterpret_cast<const uint16_t*>(s_whist);
#pragma unroll
      for (int k = 0; k < KPT; ++k) {
        if (wbase + k * 64 >= wend) continue;
        const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
        if (idx < wend) s_keys[start[kv[k] >> low] + at[k]] = kv[k];
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KPT; ++k) {
        if (wbase + k * 64 >= wend) continue;
        const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
        if (idx < wend) {
          const uint32_t key = s_keys[idx];
          const uint32_t b = key >> low;
          const int32_t lo = start[b];
          const int32_t hi = b + 1 < static_cast<uint32_t>(NP) ? start[b + 1] : n;
          int32_t to = lo;
          for (int32_t q = lo; q < hi; ++q) {
            const uint32_t o = s_keys[q];
            to += (o < key || (o == key && q < idx)) ? 1 : 0;
          }
          g[to] = key + mn;
        }
      }
      __syncthreads();
      return;
    }
    __syncthreads();
  }
  uint32_t* wh = s_whist + w * ND;
  // Pass 0 needs no stability (no earlier order to keep), so it is a plain
  // counting sort with LDS atomics over the low P0 bits, one counter per
  // word of s_whist; padding stays out of it, and the rest of the last
  // partial row is filled with it, where the stable passes keep it last.
  constexpr int PER = NB / THREADS;
  {
    for (int i = tid; i < NB; i += THREADS) s_whist[i] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      if (wbase + k * 64 >= wend) continue;
      const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
      const uint32_t d = kv[k] & (NB - 1u);
      if (idx < wend) (void)count_digit<SHARED>(&s_whist[d], d, 1u);
    }
    __syncthreads();
    uint32_t cc[PER];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      cc[j] = s_whist[tid * PER + j];
      sum += cc[j];
    }
    uint32_t all;
    uint32_t run = block_excl_scan<THREADS>(sum, s_tmp, &all);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      s_whist[tid * PER + j] = run;  // cursor per digit
      run += cc[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      if (wbase + k * 64 >= wend) continue;
      const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
      const uint32_t d = kv[k] & (NB - 1u);
      if (idx < wend) s_keys[count_digit<SHARED>(&s_whist[d], d, 1u)] = kv[k];
    }
    const int32_t pad_end = (n + 63) & ~63;  // <= CAP
    for (int i = n + tid; i < pad_end; i += THREADS) s_keys[i] = 0xffffffffu;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KPT; ++k)
      if (wbase + k * 64 < wend) kv[k] = s_keys[wbase + k * 64 + static_cast<int32_t>(lane)];
    __syncthreads();
  }
  for (int shift = P0; shift < bits; shift += P1) {
    const int nb = min(P1, bits - shift);  // bits of this pass's digit
    const uint32_t dmask = (1u << nb) - 1u;
    for (int i = tid; i < WAVES * ND; i += THREADS) s_whist[i] = 0;
    __syncthreads();
    uint32_t off[KPT];
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      if (wbase + k * 64 >= wend) continue;
      const uint32_t d = (kv[k] >> shift) & dmask;
      Differ other;
#pragma unroll
      for (int bb = 0; bb < P1; ++bb) {
        if (bb >= nb) break;
        other.bit(d, bb);
      }
      off[k] = other.rank(wh, d);
    }
    __syncthreads();
    uint32_t tot[DPT];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const int d = tid * DPT + j;
      uint32_t acc = 0;
      if (d < ND) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
          const uint32_t cw = s_whist[ww * ND + d];
          s_whist[ww * ND + d] = acc;
          acc += cw;
        }
      }
      tot[j] = acc;
      sum += acc;
    }
    uint32_t all;
    uint32_t ds = block_excl_scan<THREADS>(sum, s_tmp, &all);
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const int d = tid * DPT + j;
      if (d < ND) s_dstart[d] = ds;
      ds += tot[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      if (wbase + k * 64 >= wend) continue;
      const uint32_t d = (kv[k] >> shift) & dmask;
      s_keys[s_dstart[d] + wh[d] + off[k]] = kv[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KPT; ++k)
      if (wbase + k * 64 < wend) kv[k] = s_keys[wbase + k * 64 + static_cast<int32_t>(lane)];
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t idx = wbase + k * 64 + static_cast<int32_t>(lane);
    if (idx < wend) g[idx] = kv[k] + mn;
  }
}

}  // namespace ocp
