// Stages 1 to 6 of a small cloud in one workgroup: box, Morton codes, sort,
// unique, radix tree, edge counts and their scan, with the keys in LDS from one
// stage to the next. The same outputs as the kernels of those stages give; the
// octree kernel follows.
//
// A build of such a cloud moves next to nothing: it is launches and the round
// trips inside them, nine kernels of 4 to 11 us each. One workgroup keeps every
// array in LDS and needs neither the begin kernel nor a lookback. A build and
// its counts, us, the stages' kernels -> this one: 700 uniform points 85 -> 32,
// 4096 89 -> 47 (clustered 95 -> 60), 8192 92 -> 65 (clustered 100 -> 84); in
// batches, a workgroup per cloud: 64 x 4096 108 -> 59, 512 x 4096 199 -> 120,
// 2000 x 8192 909 -> 709.
#include "bucket_sort.hpp"
#include "pair_rows.hpp"

namespace ocp {
namespace {

constexpr int kThreads = 1024;

// Rows of 16 pairs' common prefixes, and of the minima of 16, 256 and 4096.
struct Levels {
  const v4u* row[4];
};

// The nearest position right of q (left of it) whose value is below the row
// key's, or -1. The last level is one row.
template <int TOP>
__device__ __forceinline__ int32_t next_below(const Levels& lv, uint32_t q, uint32_t key) {
  uint32_t at = q;
#pragma unroll
  for (int l = 0; l <= TOP; ++l) {
    const uint32_t hit = below16(lv.row[l][at >> 4], key) & (0xfffeu << (at & 15u)) & 0xffffu;
    if (hit) {
      at = (at & ~15u) + static_cast<uint32_t>(__builtin_ctz(hit));
#pragma unroll
      for (int d = TOP - 1; d >= 0; --d)
        if (d < l) at = at * 16u + static_cast<uint32_t>(__builtin_ctz(below16(lv.row[d][at], key)));
      return static_cast<int32_t>(at);
    }
    at >>= 4;
  }
  return -1;
}
template <int TOP>
__device__ __forceinline__ int32_t last_below(const Levels& lv, uint32_t q, uint32_t key) {
  uint32_t at = q;
#pragma unroll
  for (int l = 0; l <= TOP; ++l) {
    const uint32_t hit = below16(lv.row[l][at >> 4], key) & ((1u << (at & 15u)) - 1u);
    if (hit) {
      at = (at & ~15u) + 31u - static_cast<uint32_t>(__clz(static_cast<int>(hit)));
#pragma unroll
      for (int d = TOP - 1; d >= 0; --d)
        if (d < l)
          at = at * 16u + 31u - static_cast<uint32_t>(__clz(static_cast<int>(below16(lv.row[d][at], key))));
      return static_cast<int32_t>(at);
    }
    at >>= 4;
  }
  return -1;
}

// One workgroup per segment of at most 1024 * KPT points.
template <int KPT, bool F3>
__global__ __launch_bounds__(kThreads) void small_cloud_kernel(
    const float* __restrict__ pts, SegView sv, bool device_box, float* __restrict__ box_min,
    float* __restrict__ box_range_out, SmallOut o, uint32_t* __restrict__ ctrl) {
  constexpr int CAP = kThreads * KPT;
  constexpr int ROWS = CAP / 16;
  constexpr int TOP = CAP > 4096 ? 3 : 2;  // the level of one row
  __shared__ __attribute__((aligned(16))) uint32_t s_key[CAP];  // codes, sorted, then unique
  __shared__ v4u s_b[ROWS];
  __shared__ v4u s_b16[ROWS / 16];
  __shared__ v4u s_b256[TOP > 2 ? ROWS / 256 : 1];
  __shared__ v4u s_b4096;
  __shared__ int32_t s_edge[CAP];
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

  // ---- sort (the span is found from the keys: a small cloud may lie anywhere)
  if (n > 1) lds_bucket_sort<kThreads / 64, KPT, 12, 8, 13>(s_key, s_key, n);
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

  // ---- radix tree (k_radix_tree.hip): the pairs' common prefixes and minima
  uint8_t* b8 = reinterpret_cast<uint8_t*>(s_b);
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int32_t i = k * kThreads + tid;
    b8[i] = static_cast<uint8_t>(i < m ? clz32(s_key[i] ^ s_key[i + 1]) : 0u);
  }
  __syncthreads();
  if (tid < ROWS) reinterpret_cast<uint8_t*>(s_b16)[tid] = static_cast<uint8_t>(min16(s_b[tid]));
  __syncthreads();
  if constexpr (TOP > 2) {
    if (tid < ROWS / 16)
      reinterpret_cast<uint8_t*>(s_b256)[tid] = static_cast<uint8_t>(min16(s_b16[tid]));
    __syncthreads();
    if (tid < 16)
      reinterpret_cast<uint8_t*>(&s_b4096)[tid] =
          static_cast<uint8_t>(tid < ROWS / 256 ? min16(s_b256[tid]) : 31u);
  } else {
    if (tid < 16)
      reinterpret_cast<uint8_t*>(s_b256)[tid] =
          static_cast<uint8_t>(tid < ROWS / 16 ? min16(s_b16[tid]) : 31u);
  }
  __syncthreads();
  const Levels lv{{s_b, s_b16, s_b256, &s_b4096}};
  const uint32_t code_0 = s_key[0];
  const uint32_t b_root = m > 0 ? clz32(code_0 ^ s_key[m]) : 0u;
  const uint32_t pn_0 = m > 0 ? delta(code_0, s_key[m - 1]) : 0u;  // node 0's prefix length
#pragma unroll 1
  for (int32_t g = tid; g < m; g += kThreads) {
    const uint32_t b = b8[g];
    const uint32_t rk = __builtin_amdgcn_perm(0u, b + 127u, 0u);
    // (the position after the last pair holds 0, so the right end is found;
    // the last pair of a full array ends at m)
    int32_t r = next_below<TOP>(lv, static_cast<uint32_t>(g), rk);
    const int32_t l = last_below<TOP>(lv, static_cast<uint32_t>(g), rk);
    if (r < 0) r = m;
    const uint32_t b_l = l >= 0 ? b8[l] : 0u;
    const uint32_t b_r = r < m ? b8[r] : 0u;
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
      s_edge[node] = e;
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
      s_edge[i] = run;
      top = max(top, run + e[j]);
    }
  }
  top = wave_max(top);
  if (lane_id() == 0) atomicMax(&s_max, top);
  __syncthreads();
  for (int32_t i = tid; i < m; i += kThreads) o.offs[sb + i] = s_edge[i];
  if (tid == 0) {
    o.n_unique[seg] = u;
    o.kalloc[seg] = u > 0 ? s_max : 0;
    if (seg == 0) ctrl[kCtrlMsdTiles] = 0u;  // (an earlier build's)
  }
}

// The keys-only sort entry for few keys: one launch instead of six.
template <int WAVES, int KPT, int P0, int BINS>
__global__ __launch_bounds__(WAVES * 64) void small_sort_kernel(uint32_t* __restrict__ keys,
                                                               int32_t n,
                                                               const uint32_t* __restrict__ ctrl) {
  if (stopped_any(ctrl)) return;
  lds_bucket_sort<WAVES, KPT, P0, 8, BINS>(keys, keys, n);
}

}  // namespace

void launch_small_sort(uint32_t* keys, int32_t n, const uint32_t* ctrl, hipStream_t s) {
  if (n <= 4096)
    small_sort_kernel<16, 4, 12, 13><<<1, 1024, 0, s>>>(keys, n, ctrl);
  else
    small_sort_kernel<16, 16, 12, 13><<<1, 1024, 0, s>>>(keys, n, ctrl);
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
