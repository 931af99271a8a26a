// Stages 1 to 6 of a small cloud in one workgroup: box, Morton codes, sort,
// unique, radix tree, edge counts and their scan, with the keys in LDS from one
// stage to the next. The same outputs as the kernels of those stages give; the
// octree kernel follows.
//
// A build of such a cloud moves next to nothing: it is launches and the round
// trips inside them, nine kernels of 4 to 11 us each. One workgroup keeps every
// array in LDS and needs neither the begin kernel nor a lookback. A build and
// its counts, us, the stages' kernels -> this one: 700 uniform points 85 -> 27,
// 4096 89 -> 36 (clustered 95 -> 48), 8192 92 -> 49 (clustered 100 -> 63); in
// batches, a workgroup per cloud: 64 x 4096 108 -> 47, 512 x 4096 199 -> 87,
// 2000 x 8192 909 -> 545.
#include "bucket_sort.hpp"

namespace ocp {
namespace {

constexpr int kThreads = 1024;

// Which pairs' common prefix is below b, for each b: a row of 64-bit words a
// value (a word more than it has, so that one word's values lie in different
// banks), and which words of it are not zero. A pair's nearest ones below its own
// are then a few bit operations on one or two words on either side. (Against
// walks over rows of 16 bytes and their minima, which took 19,000 of 8192 points'
// 81,000 cycles a side: 4096 points 40.4 -> 36.8 us, 8192 56.7 -> 49.5.)
template <int WORDS>
struct Below {
  static constexpr int kStride = WORDS + 1;
  uint64_t low[32 * kStride];
  uint64_t any[32][WORDS / 64];

  // The nearest position right of g; there is one.
  __device__ __forceinline__ int32_t next(int32_t g, uint32_t b, uint64_t word) const {
    uint32_t w = static_cast<uint32_t>(g) >> 6;
    uint64_t hit = word & (~1ull << (g & 63));
    if (!hit) {
      uint64_t rest = any[b][w >> 6] & (~1ull << (w & 63u));
      if (WORDS > 64 && !rest && w < 64u) {
        rest = any[b][WORDS / 64 - 1];
        w = 64u;
      }
      w = (w & ~63u) + static_cast<uint32_t>(__builtin_ctzll(rest));
      hit = low[b * kStride + w];
    }
    return static_cast<int32_t>(w * 64u) + __builtin_ctzll(hit);
  }
  // The nearest left of g, or -1.
  __device__ __forceinline__ int32_t last(int32_t g, uint32_t b, uint64_t word) const {
    uint32_t w = static_cast<uint32_t>(g) >> 6;
    uint64_t hit = word & ((1ull << (g & 63)) - 1ull);
    if (!hit) {
      uint64_t rest = any[b][w >> 6] & ((1ull << (w & 63u)) - 1ull);
      if (WORDS > 64 && !rest && w >= 64u) {
        rest = any[b][0];
        w = 0u;
      }
      if (!rest) return -1;
      w = (w & ~63u) + 63u - static_cast<uint32_t>(__builtin_clzll(rest));
      hit = low[b * kStride + w];
    }
    return static_cast<int32_t>(w * 64u) + 63 - __builtin_clzll(hit);
  }
};

// One workgroup per segment of at most 1024 * KPT points.
template <int KPT, bool F3>
__global__ __launch_bounds__(kThreads) void small_cloud_kernel(
    const float* __restrict__ pts, SegView sv, bool device_box, float* __restrict__ box_min,
    float* __restrict__ box_range_out, SmallOut o, uint32_t* __restrict__ ctrl) {
  constexpr int CAP = kThreads * KPT;
  constexpr int WORDS = CAP / 64;
  static_assert(WORDS == 64 || WORDS == 128, "one or two words say which words of a row count");
  __shared__ __attribute__((aligned(16))) uint32_t s_key[CAP];  // codes, sorted, then unique
  __shared__ uint8_t s_b[CAP];  // the pairs' common prefixes
  __shared__ Below<WORDS> s_below;
  __shared__ int8_t s_edge[CAP];  // (at most 10 levels)
  __shared__ uint32_t s_tmp[kThreads / 64];
  __shared__ uint32_t s_box[2];
  __shared__ int32_t s_max;
  const int tid = threadIdx.x;
  const int32_t seg = blockIdx.x;
  const int32_t sb = seg_begin(sv, seg);
  const int32_t n = seg_end(sv, seg) - sb;
  if (stopped_any(ctrl)) {
    // (an earlier build's time-out, not yet reported: no keys, no slots)
    if (tid == 0) {
      o.n_unique[seg] = 0;
      o.kalloc[seg] = 0;
    }
    return;
  }

  for (int i = tid; i < 32 * (WORDS + 1); i += kThreads) s_below.low[i] = 0u;

  // ---- points, box, codes
  float x[KPT], y[KPT], z[KPT];
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t i = k * kThreads + tid;
    x[k] = y[k] = z[k] = 0.0f;
    if (i < n) {
      const int64_t g = static_cast<int64_t>(sb) + i;
      if constexpr (F3) {
        x[k] = pts[3 * g];
        y[k] = pts[3 * g + 1];
        z[k] = pts[3 * g + 2];
      } else {
        const float4 p = reinterpret_cast<const float4*>(pts)[g];
        x[k] = p.x;
        y[k] = p.y;
        z[k] = p.z;
      }
    }
  }
  float mn, rg;
  if (device_box) {
    if (tid == 0) {
      s_box[0] = 0xffffffffu;
      s_box[1] = 0u;
    }
    __syncthreads();
    uint32_t lo = 0xffffffffu, hi = 0u;
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      if (k * kThreads + tid >= n) continue;
      const uint32_t a = ord(x[k]), b = ord(y[k]), c = ord(z[k]);
      lo = min(lo, min(a, min(b, c)));
      hi = max(hi, max(a, max(b, c)));
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    if (lane_id() == 0) {
      atomicMin(&s_box[0], lo);
      atomicMax(&s_box[1], hi);
    }
    __syncthreads();
    const bool none = s_box[0] > s_box[1];  // an empty cloud gets (0, 1)
    mn = none ? 0.0f : unord(s_box[0]);
    rg = none ? 1.0f : box_range(mn, unord(s_box[1]));
    if (tid == 0) {
      box_min[seg] = mn;
      box_range_out[seg] = rg;
    }
  } else {
    mn = seg_min(sv, seg);
    rg = seg_range(sv, seg);
  }
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t i = k * kThreads + tid;
    if (i < n) s_key[i] = encode(x[k], y[k], z[k], mn, rg);
  }
  if (tid == 0) s_max = 1;
  __syncthreads();

  // ---- sort (the span is found from the keys: a small cloud may lie anywhere).
  // Crowded keys take stable passes after the first 12 bits: where one workgroup
  // fits a CU anyway, of 9 bits, two for 30 bits and not three (8192 clustered
  // points 65.7 -> 63.4 us a build; at 4096 points the counters would cost the
  // second workgroup).
  if (n > 1) lds_bucket_sort<kThreads / 64, KPT, 12, (KPT > 4 ? 9 : 8), 13>(s_key, s_key, n);
  __syncthreads();

  // ---- unique: thread t holds keys t*KPT .. t*KPT + KPT-1
  uint32_t key[KPT];
  uint32_t keep = 0;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int32_t i = tid * KPT + j;
    key[j] = i < n ? s_key[i] : 0u;
  }
  const uint32_t prev = tid > 0 && tid * KPT <= n ? s_key[tid * KPT - 1] : 0u;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int32_t i = tid * KPT + j;
    if (i < n && (i == 0 || key[j] != (j ? key[j - 1] : prev))) keep |= 1u << j;
  }
  for (int32_t i = tid; i < n; i += kThreads) o.sorted[sb + i] = s_key[i];
  uint32_t u_total;
  uint32_t pos = block_excl_scan<kThreads>(static_cast<uint32_t>(__popc(keep)), s_tmp, &u_total);
#pragma unroll
  for (int j = 0; j < KPT; ++j)
    if ((keep >> j) & 1u) s_key[pos++] = key[j];
  __syncthreads();
  const int32_t u = static_cast<int32_t>(u_total);
  const int32_t m = u - 1;  // pairs
  for (int32_t i = tid; i < u; i += kThreads) o.unique[sb + i] = s_key[i];

  // ---- radix tree (k_radix_tree.hip): the pairs' common prefixes, where each
  // value is, then where any below it is. The position after the last pair
  // holds 0: every pair has a lower one on its right.
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t i = k * kThreads + tid;
    if (i > m) continue;
    const uint32_t b = i < m ? clz32(s_key[i] ^ s_key[i + 1]) : 0u;
    s_b[i] = static_cast<uint8_t>(b);
    atomicOr(reinterpret_cast<uint32_t*>(&s_below.low[b * (WORDS + 1) + (i >> 6)]) + ((i >> 5) & 1),
             1u << (i & 31));
  }
  __syncthreads();
  {
    const int v0 = 2 * static_cast<int>(wave_id());  // 16 waves, two values each
    uint64_t even[WORDS / 64], odd[WORDS / 64];
#pragma unroll
    for (int c = 0; c < WORDS / 64; ++c) {
      const uint64_t* at = s_below.low + c * 64 + static_cast<int>(lane_id());
      even[c] = 0u;
#pragma unroll 4
      for (int v = 0; v < v0; ++v) even[c] |= at[v * (WORDS + 1)];
      odd[c] = even[c] | at[v0 * (WORDS + 1)];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < WORDS / 64; ++c) {
      uint64_t* at = s_below.low + c * 64 + static_cast<int>(lane_id());
      at[v0 * (WORDS + 1)] = even[c];
      at[(v0 + 1) * (WORDS + 1)] = odd[c];
      const uint64_t any_even = __ballot(even[c] != 0u), any_odd = __ballot(odd[c] != 0u);
      if (lane_id() == 0) {
        s_below.any[v0][c] = any_even;
        s_below.any[v0 + 1][c] = any_odd;
      }
    }
  }
  __syncthreads();
  const uint32_t code_0 = s_key[0];
  const uint32_t b_root = m > 0 ? clz32(code_0 ^ s_key[m]) : 0u;
  const uint32_t pn_0 = m > 0 ? delta(code_0, s_key[m - 1]) : 0u;  // node 0's prefix length
#pragma unroll 1
  for (int32_t g = tid; g < m; g += kThreads) {
    const uint32_t b = s_b[g];
    const uint64_t word = s_below.low[b * (WORDS + 1) + (static_cast<uint32_t>(g) >> 6)];
    const int32_t r = s_below.next(g, b, word);
    const int32_t l = s_below.last(g, b, word);
    const uint32_t b_l = l >= 0 ? s_b[l] : 0u;
    const uint32_t b_r = s_b[r];
    const uint32_t b_up = max(b_l, b_r);
    const int32_t node = b_l >= b_r ? l + 1 : r;
    const bool leaf_l = l + 1 == g, leaf_r = r == g + 1;
    if (b_up != 0) {  // (the true root's record is node 0's, below)
      const int32_t e = static_cast<int32_t>(third(b - 1u)) -
                        static_cast<int32_t>(third(b_up == b_root ? pn_0 : b_up - 1u));
      o.prefix[sb + node] = static_cast<uint8_t>(b - 1u);
      o.hl[sb + node] = leaf_l;
      o.hr[sb + node] = leaf_r;
      o.lc[sb + node] = g;
      s_edge[node] = static_cast<int8_t>(e);
    }
    if (!leaf_l) o.par[sb + g] = node;
    if (!leaf_r) o.par[sb + g + 1] = node;
  }
  if (wave_id() == 0 && m > 0) {
    // Node 0: the range [0, m - 1] and the last s in it with a longer prefix
    // (prefixes with code_0 only get shorter: 64 probes of the rest at a time).
    int32_t lo = 1, hi = m - 1;  // the first that has none is in [lo, hi]
    while (lo < hi) {
      const int32_t step = (hi - lo + 63) >> 6;
      const int32_t at = lo + static_cast<int32_t>(lane_id()) * step;
      const int32_t has =
          __popcll(__ballot(at < hi && delta(code_0, s_key[min(at, m)]) > pn_0));
      if (has == 0) break;
      hi = min(hi, lo + has * step);
      lo += (has - 1) * step + 1;
    }
    const int32_t s = max(lo - 1, 0);
    if (lane_id() == 0) {
      o.prefix[sb] = static_cast<uint8_t>(pn_0);
      o.hl[sb] = s == 0;
      o.hr[sb] = s + 1 == m - 1;
      o.lc[sb] = s;
      o.par[sb] = 0;
      s_edge[0] = 0;
    }
  }
  __syncthreads();

  // ---- edge counts, their inclusive scan, the octree's slots
  static_assert(sizeof(s_below.low) >= sizeof(int32_t) * CAP, "the scan takes the rows' place");
  int32_t* s_run = reinterpret_cast<int32_t*>(s_below.low);
  int32_t e[KPT];
  int32_t sum = 0;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int32_t i = tid * KPT + j;
    e[j] = i < m ? s_edge[i] : 0;
    sum += e[j];
  }
  uint32_t total;
  int32_t run = static_cast<int32_t>(block_excl_scan<kThreads>(static_cast<uint32_t>(sum), s_tmp, &total));
  int32_t top = 1;
  for (int32_t i = tid; i < m; i += kThreads) o.edge[sb + i] = s_edge[i];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int32_t i = tid * KPT + j;
    run += e[j];
    if (i < m) {
      s_run[i] = run;
      top = max(top, run + e[j]);
    }
  }
  top = wave_max(top);
  if (lane_id() == 0) atomicMax(&s_max, top);
  __syncthreads();
  for (int32_t i = tid; i < m; i += kThreads) o.offs[sb + i] = s_run[i];
  if (tid == 0) {
    o.n_unique[seg] = u;
    o.kalloc[seg] = u > 0 ? s_max : 0;
    if (seg == 0) ctrl[kCtrlMsdTiles] = 0u;  // (an earlier build's)
  }
}

// The keys-only sort entry for few keys: one launch instead of six. 16,384 spread
// keys take 19 us (the passes 46). Crowded ones take the radix passes: two of 9 bits
// after 14, for which this one workgroup has the LDS. Above 8192 keys those that
// are equal in the bits of a pass are counted together: keys of a few values in the
// top bits 66 -> 41 us (the passes 44) for 19 -> 19.4 with spread ones; 8192 take
// 37 without.
template <int WAVES, int KPT, int P0, int P1, int BINS, bool SHARED>
__global__ __launch_bounds__(WAVES * 64) void small_sort_kernel(uint32_t* __restrict__ keys,
                                                               int32_t n,
                                                               const uint32_t* __restrict__ ctrl) {
  if (stopped_any(ctrl)) return;
  lds_bucket_sort<WAVES, KPT, P0, P1, BINS, SHARED>(keys, keys, n);
}

}  // namespace

void launch_small_sort(uint32_t* keys, int32_t n, const uint32_t* ctrl, hipStream_t s) {
  if (n <= 4096)
    small_sort_kernel<16, 4, 12, 8, 13, false><<<1, 1024, 0, s>>>(keys, n, ctrl);
  else if (n <= 8192)
    small_sort_kernel<16, 8, 14, 9, 13, false><<<1, 1024, 0, s>>>(keys, n, ctrl);
  else
    small_sort_kernel<16, 16, 14, 9, 13, true><<<1, 1024, 0, s>>>(keys, n, ctrl);
}

void launch_small_clouds(const float* pts, bool float3, const SegView& sv, int64_t max_seg,
                         bool device_boxes, float* box_min, float* box_range, const SmallOut& o,
                         uint32_t* ctrl, hipStream_t s) {
  if (sv.n_seg <= 0) return;
  const auto go = [&](auto kernel) {
    kernel<<<sv.n_seg, kThreads, 0, s>>>(pts, sv, device_boxes, box_min, box_range, o, ctrl);
  };
  if (max_seg <= 4096) {
    if (float3) go(small_cloud_kernel<4, true>);
    else go(small_cloud_kernel<4, false>);
  } else {
    if (float3) go(small_cloud_kernel<8, true>);
    else go(small_cloud_kernel<8, false>);
  }
}

}  // namespace ocp
