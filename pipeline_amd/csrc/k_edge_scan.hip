// Stage 5 (kernels/05_edge_count.cpp:3-16: e[0] = 0, e[i] = prefix_n[i]/3 -
// prefix_n[parent[i]]/3) for the per-stage entry, and stage 6: the inclusive
// scan of kernels/06_partial_sum.cpp:3-15 (the reference GPU path has no scan
// and round-trips to the host, apps/gpu_demo/main.cu:308-310). In the fused
// build the radix-tree kernel writes the edge counts.
//
// The scan: tiles of 256*IPT entries, one per workgroup, one lookback chain
// per segment. A thread takes four consecutive entries per row of 1024 (one
// 16-byte load and store; the sums of the four are scanned, a quarter of the
// wave scans of one entry per lane); one wave scans the IPT row totals and
// does the two-level lookback (the tile's group of 64, then the sums of
// earlier groups). The tiles' maxima of P[i] + e[i] reach the segment's
// octree slot count with one atomicMax per group of 64 tiles.
#include "ocp_internal.hpp"

namespace ocp {
namespace {

typedef int32_t v4i __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void edge_count_kernel(const uint8_t* __restrict__ prefix_n,
                                                         const int32_t* __restrict__ parent,
                                                         int32_t* __restrict__ edge, int32_t n,
                                                         const uint32_t* __restrict__ ctrl) {
  if (stopped_any(ctrl)) return;
  const int32_t i = static_cast<int32_t>(blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  int32_t v = 0;
  if (i > 0)
    v = static_cast<int32_t>(static_cast<uint32_t>(prefix_n[i]) / 3) -
        static_cast<int32_t>(static_cast<uint32_t>(prefix_n[parent[i]]) / 3);
  edge[i] = v;
}

template <int IPT>
__global__ __launch_bounds__(256) void edge_scan_kernel(
    const int32_t* __restrict__ edge_all, int32_t* __restrict__ off_all, SegView sv,
    const int32_t* __restrict__ tile_start, const int32_t* __restrict__ n_unique, int32_t n_host,
    uint64_t* __restrict__ flags, uint32_t* __restrict__ ctrl, int32_t* __restrict__ kalloc) {
  constexpr int THREADS = 256;
  constexpr int NW = THREADS / 64;
  constexpr int T = THREADS * IPT;
  constexpr int ROWS = IPT / 4;
  __shared__ uint32_t s_rows[ROWS * NW];
  __shared__ int32_t s_max[NW];
  __shared__ uint32_t s_excl;

  const int tid = threadIdx.x;
  const uint32_t w = wave_id();
  const uint32_t lane = lane_id();
  const int32_t t = blockIdx.x;  // in-order dispatch: see lookback_n
  const uint32_t tag = ctrl[kCtrlEpoch] * 8u + kStageScan;
  if (stopped(ctrl, tag)) return;
  const TileRef r = find_tile(tile_start, sv.n_seg, t);
  const int32_t n = n_unique ? n_unique[r.seg] - 1 : n_host;
  const int32_t sb = seg_begin(sv, r.seg);  // loaded with n, before the test
  const int32_t base = r.local * T;
  if (base >= n) return;  // no later tile of this chain waits on it
  const int32_t cnt = min(T, n - base);
  const int32_t* edge = edge_all + sb + base;
  int32_t* off = off_all + sb + base;

  // Loads first, all in flight together (4-byte aligned: a segment or a
  // caller's range starts anywhere).
  v4i e[ROWS];
  if (cnt == T) {
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
      __builtin_memcpy(&e[k], edge + k * 1024 + tid * 4, 16);
  } else {
#pragma unroll
    for (int k = 0; k < ROWS; ++k) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int32_t idx = k * 1024 + tid * 4 + u;
        e[k][u] = idx < cnt ? edge[idx] : 0;
      }
    }
  }
  uint32_t before[ROWS];  // sum of the row's earlier lanes in this wave
#pragma unroll
  for (int k = 0; k < ROWS; ++k) {
    const uint32_t sum = static_cast<uint32_t>(e[k].x) + static_cast<uint32_t>(e[k].y) +
                         static_cast<uint32_t>(e[k].z) + static_cast<uint32_t>(e[k].w);
    const uint32_t incl = wave_incl_scan(sum);
    before[k] = incl - sum;
    if (lane == 63) s_rows[k * NW + w] = incl;
  }
  __syncthreads();
  if (w == 0) {
    const uint32_t total = wave_scan_lds<ROWS * NW>(s_rows);
    if (lane == 0)
      flag_store(&flags[t], flag_pack(tag, kFlagAgg, total));
    bool late = false;
    // Group sums live after the grid's tile flags.
    const uint32_t prev =
        wave_lookback_groups(flags, flags + gridDim.x, t, t - r.local, total, tag,
                             wait_limit(ctrl), &late);
    if (lane == 0) {
      if (late) raise_timeout(ctrl, tag);
      s_excl = prev;
    }
  }
  __syncthreads();
  const uint32_t excl = s_excl;
  int32_t kmax = 1;
  uint32_t rb[ROWS];  // all LDS reads before the stores
#pragma unroll
  for (int k = 0; k < ROWS; ++k) rb[k] = s_rows[k * NW + w];
#pragma unroll
  for (int k = 0; k < ROWS; ++k) {
    v4i p;
    uint32_t run = excl + rb[k] + before[k];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      run += static_cast<uint32_t>(e[k][u]);
      p[u] = static_cast<int32_t>(run);
    }
    const int32_t idx = k * 1024 + tid * 4;
    if (idx + 4 <= cnt) {
      __builtin_memcpy(off + idx, &p, 16);
#pragma unroll
      for (int u = 0; u < 4; ++u) kmax = max(kmax, p[u] + e[k][u]);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (idx + u < cnt) {
          off[idx + u] = p[u];
          kmax = max(kmax, p[u] + e[k][u]);
        }
      }
    }
  }
  if (kalloc) {
    kmax = wave_max(kmax);
    if (lane == 0) s_max[w] = kmax;
    __syncthreads();
    if (w == 0) {
      int32_t m = s_max[0];
#pragma unroll
      for (int q = 1; q < NW; ++q) m = max(m, s_max[q]);
      // Tile maxima reach K_alloc one group of 64 tiles at a time: the last
      // tile of a group (or of the segment) folds in the maxima its group's
      // earlier tiles published, so the segment's counter takes one atomic
      // per group (same-address atomics from every tile serialise: 19 us at
      // 10M). The waits go to earlier tiles only.
      uint64_t* mflags = flags + 2 * static_cast<int64_t>(gridDim.x);
      if (lane == 0) flag_store(mflags + t, flag_pack(tag, kFlagAgg, static_cast<uint32_t>(m)));
      const int32_t local = r.local;
      const int32_t g0 = local & ~63;
      if ((local & 63) == 63 || local == (n + T - 1) / T - 1) {
        bool late = false;
        const uint32_t gm = wave_sum_flags<true>(mflags + (t - local) + g0, 1, local - g0,
                                                 tag & 0x3fffffffu, wait_limit(ctrl), &late);
        if (lane == 0) {
          if (late) raise_timeout(ctrl, tag);
          atomicMax(&kalloc[r.seg], max(m, static_cast<int32_t>(gm)));
        }
      }
    }
  }
}

}  // namespace

void launch_edge_count(const uint8_t* prefix_n, const int32_t* parent, int32_t* edge, int32_t n,
                       const uint32_t* ctrl, hipStream_t s) {
  if (n <= 0) return;
  edge_count_kernel<<<(n + 255) / 256, 256, 0, s>>>(prefix_n, parent, edge, n, ctrl);
}

void launch_edge_scan(const int32_t* edge, int32_t* offsets, const SegView& sv,
                      const int32_t* tile_start, int32_t total_tiles, const int32_t* n_unique,
                      int32_t n_host, uint64_t* flags, uint32_t* ctrl, int32_t* kalloc,
                      const TuneTable& tt, hipStream_t s) {
  if (total_tiles <= 0) return;
  const auto go = [&](auto kernel) {
    kernel<<<total_tiles, 256, 0, s>>>(edge, offsets, sv, tile_start, n_unique, n_host, flags,
                                       ctrl, kalloc);
  };
  switch (tt.scan_ipt) {
    case 32: go(edge_scan_kernel<32>); break;
    case 8: go(edge_scan_kernel<8>); break;
    default: go(edge_scan_kernel<16>); break;
  }
}

}  // namespace ocp
