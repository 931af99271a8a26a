// MSD form of a build's sort (bare 30-bit Morton keys). One scatter by the top
// 10-bit digit (bits 20-29; cursor_scatter.hpp, no lookback: the order within
// a digit is free) leaves the keys of every top digit contiguous, and windows
// of them are sorted in LDS (bucket_sort.hpp). The result is the sorted key
// array, the same bytes as the LSD passes of kernels/02_sort.cpp:5-118 give.
//
// A window is the digits whose keys start in it, so the LDS sorts are alike
// however the keys are spread. A digit with more keys than the LDS holds is
// left to a second level, three kernels that return at once when there is no
// such digit: the counts of the next 10 bits over the digit's keys, a scatter
// by them into the other buffer, and again windows of the result, sorted back
// into place. A second-level digit holds one 20-bit prefix; one with more
// keys than the LDS holds is written from the counts of its low 10 bits, by
// the workgroup of its first window, or, above kShare keys, by those of all
// its windows from counts that the second scatter takes along.
//
// No kernel waits for another workgroup, and the passes over memory are two
// for keys of ordinary digits and four (a read of them, two scatters, the
// windows) for the others, against four passes and their lookbacks. At 10M
// uniform points: scatter 35 us, windows 44 (58 before the binning of
// bucket_sort.hpp), the idle second level 14, against 38 + 3 x 45 us for four
// 8-bit passes; 2^24 clustered points, most of whose keys take the second level:
// scatter 38, windows 27, then counts 28, scatter 36 and windows 104 us, against
// 250. The LDS sorts bound it: 2 (8) waves a SIMD by LDS, and their chain of
// barriers. Figures of whole builds are given at the rule that takes this form,
// beside auto_sort_msd.
#include "bucket_sort.hpp"
#include "cursor_scatter.hpp"

namespace ocp {
namespace {

constexpr int kRadix = 1024;
constexpr int kL2Tile = 8192;           // keys per second-level tile and window
constexpr uint32_t kShare = 65536;      // keys of one 20-bit prefix that a workgroup writes alone

struct MiddleDigit10 {
  static constexpr bool kCheap = true;
  static constexpr int kBits = 10;
  __device__ __forceinline__ uint32_t operator()(uint32_t key) const {
    return (key >> 10) & 1023u;
  }
};

// The digits whose keys start in window [wlo, whi) of a segment, from the
// segment's 1024 counts; with only >= 0 that digit alone. Offsets are relative
// to the segment.
struct Window {
  uint32_t first, last;  // first and last nonempty digit that starts in it
  uint32_t a, c0, b;     // start of first, start of last, end of last
  uint32_t cont, cont_start, cont_end;  // the digit that reaches in from before
  bool any, reaches;
};

template <int THREADS>
__device__ __forceinline__ Window find_window(const uint32_t* __restrict__ counts, int32_t only,
                                              uint32_t wlo, uint32_t whi,
                                              uint32_t (&cnt)[kRadix / THREADS]) {
  constexpr int PER = kRadix / THREADS;
  __shared__ uint32_t s_tmp[THREADS / 64];
  __shared__ uint32_t s_w[8];
  const int tid = threadIdx.x;
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) cnt[j] = counts[tid * PER + j];
#pragma unroll
  for (int j = 0; j < PER; ++j) sum += cnt[j];
  if (tid < 8) s_w[tid] = tid == 0 ? kRadix : 0u;
  uint32_t total;
  uint32_t st = block_excl_scan<THREADS>(sum, s_tmp, &total);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t d = static_cast<uint32_t>(tid * PER + j);
    const uint32_t en = st + cnt[j];
    if (cnt[j] && (only >= 0 ? d == static_cast<uint32_t>(only) : st >= wlo && st < whi)) {
      atomicMin(&s_w[0], d);
      atomicMax(&s_w[1], d + 1);
    }
    if (cnt[j] && st < wlo && en > wlo) {
      s_w[2] = d;
      s_w[3] = st;
      s_w[4] = en;
    }
    st = en;
  }
  __syncthreads();
  st -= sum;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t d = static_cast<uint32_t>(tid * PER + j);
    if (d == s_w[0]) s_w[5] = st;
    if (d + 1 == s_w[1]) {
      s_w[6] = st;
      s_w[7] = st + cnt[j];
    }
    st += cnt[j];
  }
  __syncthreads();
  Window w;
  w.any = s_w[1] != 0;
  w.first = s_w[0];
  w.last = s_w[1] - 1u;
  w.a = s_w[5];
  w.c0 = s_w[6];
  w.b = s_w[7];
  w.reaches = s_w[4] != 0;
  w.cont = s_w[2];
  w.cont_start = s_w[3];
  w.cont_end = s_w[4];
  return w;
}

// Bits that the keys of n neighbouring digits of `low` bits each span.
__device__ __forceinline__ int span_bits(uint32_t n, int low) {
  return low + (n > 1 ? 32 - __clz(static_cast<int>(n - 1)) : 0);
}

// First level: window `local` of a segment (of a long one the digit of that
// number, see msd_window), sorted in place. A digit above CAP is listed for the
// second level, with its counts and cursors cleared.
// (four waves a SIMD: what the LDS of the larger workgroups allows)
template <int WAVES, int KPT, int P1, int BINS>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(4))) void msd_window_kernel(
    uint32_t* __restrict__ keys, SegView sv, const int32_t* __restrict__ tile_start,
    const uint32_t* __restrict__ hist, MsdLevel2 l2, uint32_t* __restrict__ ctrl) {
  constexpr int THREADS = WAVES * 64;
  constexpr uint32_t CAP = THREADS * KPT;
  __shared__ int32_t s_big[3];
  if (stopped_any(ctrl)) return;
  const TileRef r = find_tile(tile_start, sv.n_seg, static_cast<int32_t>(blockIdx.x));
  const int32_t sb = seg_begin(sv, r.seg);
  const int32_t len = seg_end(sv, r.seg) - sb;
  const int32_t window = msd_window(WAVES == 4, len);
  const uint32_t wlo = static_cast<uint32_t>(r.local) * static_cast<uint32_t>(window);
  uint32_t cnt[kRadix / THREADS];
  const Window w = find_window<THREADS>(
      hist + static_cast<int64_t>(r.seg) * hist_stride(10) + 2 * kRadix, window ? -1 : r.local, wlo,
      min(wlo + static_cast<uint32_t>(window), static_cast<uint32_t>(len)), cnt);
  // (counts that do not describe the segment cannot come from its Morton
  // kernel; nothing outside it is touched then)
  if (!w.any || w.b > static_cast<uint32_t>(len)) return;
  uint32_t* seg = keys + sb;
  if (w.b - w.a <= CAP) {
    if (w.b - w.a > 1)
      lds_bucket_sort<WAVES, KPT, 12, P1, BINS>(seg + w.a, seg + w.a,
                                                static_cast<int32_t>(w.b - w.a), w.first << 20,
                                                span_bits(w.last - w.first + 1u, 20));
    return;
  }
  // (not in a loop: the compiler would keep every row's addresses across it)
  if (w.c0 - w.a > 1)
    lds_bucket_sort<WAVES, KPT, 12, P1, BINS>(seg + w.a, seg + w.a,
                                              static_cast<int32_t>(w.c0 - w.a), w.first << 20,
                                              span_bits(w.last - w.first, 20));
  const uint32_t n = w.b - w.c0;
  if (n <= CAP) {
    if (n > 1)
      lds_bucket_sort<WAVES, KPT, 12, P1, BINS>(seg + w.c0, seg + w.c0, static_cast<int32_t>(n),
                                                w.last << 20, 20);
    return;
  }
  const int32_t tiles = static_cast<int32_t>((n + kL2Tile - 1) / kL2Tile);
  const int tid = threadIdx.x;
  if (tid == 0) {
    s_big[0] = static_cast<int32_t>(atomicAdd(&ctrl[kCtrlMsdBig], 1u));
    s_big[1] = static_cast<int32_t>(atomicAdd(&ctrl[kCtrlMsdTiles], static_cast<uint32_t>(tiles)));
    s_big[2] = static_cast<int32_t>(atomicAdd(&ctrl[kCtrlMsdSlots], n / kShare));
  }
  __syncthreads();
  const int32_t big = s_big[0], t0 = s_big[1];
  if (big >= l2.max_big || t0 + tiles > l2.max_tiles) return;  // (never: sized for any keys)
  if (tid == 0)
    l2.big[big] = make_int4(sb + static_cast<int32_t>(w.c0), static_cast<int32_t>(n),
                            static_cast<int32_t>(w.last), s_big[2]);
  for (int32_t k = tid; k < tiles; k += THREADS) l2.tiles[t0 + k] = make_int2(big, k);
  for (int k = tid; k < kRadix; k += THREADS) {
    l2.hist[static_cast<int64_t>(big) * kRadix + k] = 0;
    l2.cursor[static_cast<int64_t>(big) * kRadix + k] = 0;
  }
}

// Second level: counts of bits 10-19 over the listed digits' keys.
__global__ __launch_bounds__(512) void msd_l2_hist_kernel(const uint32_t* __restrict__ keys,
                                                          MsdLevel2 l2,
                                                          const uint32_t* __restrict__ ctrl) {
  __shared__ uint32_t s_hist[kRadix];
  const int32_t n_tiles = static_cast<int32_t>(ctrl[kCtrlMsdTiles]);
  if (n_tiles == 0 || stopped_any(ctrl)) return;
  const int tid = threadIdx.x;
  const int64_t slots = min(static_cast<int64_t>(ctrl[kCtrlMsdSlots]), static_cast<int64_t>(l2.max_slots));
  for (int64_t k = blockIdx.x * 512 + tid; k < slots * kRadix; k += gridDim.x * 512) l2.hist3[k] = 0;
  for (int32_t t = blockIdx.x; t < n_tiles; t += gridDim.x) {
    for (int k = tid; k < kRadix; k += 512) s_hist[k] = 0;
    __syncthreads();
    const int2 ref = l2.tiles[t];
    const int4 big = l2.big[ref.x];
    const int32_t base = ref.y * kL2Tile;
    const int32_t cnt = min(kL2Tile, big.y - base);
    const uint32_t* src = keys + big.x + base + tid;
    uint32_t v[kL2Tile / 512];
#pragma unroll
    for (int k = 0; k < kL2Tile / 512; ++k) v[k] = k * 512 + tid < cnt ? src[k * 512] : 0u;
#pragma unroll
    for (int k = 0; k < kL2Tile / 512; ++k)
      if (k * 512 + tid < cnt) atomicAdd(&s_hist[(v[k] >> 10) & 1023u], 1u);
    __syncthreads();
    for (int k = tid; k < kRadix; k += 512)
      if (s_hist[k]) atomicAdd(&l2.hist[static_cast<int64_t>(ref.x) * kRadix + k], s_hist[k]);
    __syncthreads();
  }
}

// The number of this workgroup's digits before `digit` with more than kShare
// keys, one digit per thread.
__device__ __forceinline__ uint32_t shared_before(uint32_t n, uint32_t digit, uint32_t* s) {
  __syncthreads();
  if (threadIdx.x == 0) *s = 0;
  __syncthreads();
  if (n > kShare && threadIdx.x < digit) atomicAdd(s, 1u);
  __syncthreads();
  return *s;
}

// ... their scatter by those bits, into the other buffer. The keys of a digit
// above kShare also count their low 10 bits.
__global__ __launch_bounds__(1024) void msd_l2_scatter_kernel(const uint32_t* __restrict__ in,
                                                              uint32_t* __restrict__ out,
                                                              MsdLevel2 l2,
                                                              const uint32_t* __restrict__ ctrl) {
  __shared__ uint32_t s_low[kRadix];
  __shared__ uint32_t s_n;
  __shared__ uint32_t s_rank;
  const int32_t n_tiles = static_cast<int32_t>(ctrl[kCtrlMsdTiles]);
  if (n_tiles == 0 || stopped_any(ctrl)) return;
  const uint32_t tid = threadIdx.x;
  const int32_t t = blockIdx.x;
  if (t >= n_tiles) return;
  const int2 ref = l2.tiles[t];
  const int4 big = l2.big[ref.x];
  const int32_t base = ref.y * kL2Tile;
  const int32_t cnt = min(kL2Tile, big.y - base);
  const auto count_low = [&](uint32_t n, const uint32_t (&dg)[kL2Tile / 1024],
                             const uint32_t (&keys)[kL2Tile / 1024]) {
    if (!__syncthreads_or(n > kShare)) return;
    for (uint32_t d = 0; d < kRadix; ++d) {
      // (uniform: the next digit above kShare, through LDS)
      __syncthreads();
      if (tid == 0) s_n = kRadix;
      s_low[tid] = 0;
      __syncthreads();
      if (n > kShare && tid >= d) atomicMin(&s_n, tid);
      __syncthreads();
      d = s_n;
      if (d >= kRadix) break;
      const uint32_t slot = static_cast<uint32_t>(big.w) + shared_before(n, d, &s_rank);
#pragma unroll
      for (int k = 0; k < kL2Tile / 1024; ++k)
        if (dg[k] == d) atomicAdd(&s_low[keys[k] & 1023u], 1u);
      __syncthreads();
      if (s_low[tid] && slot < static_cast<uint32_t>(l2.max_slots))
        atomicAdd(&l2.hist3[static_cast<int64_t>(slot) * kRadix + tid], s_low[tid]);
    }
    __syncthreads();
  };
  cursor_scatter_tile<1024, kL2Tile / 1024>(
      in, out, big.x, big.y, big.x + base, cnt, l2.hist + static_cast<int64_t>(ref.x) * kRadix,
      l2.cursor + static_cast<int64_t>(ref.x) * kRadix, MiddleDigit10{}, count_low);
}

// Positions [from, to) of the run of one 20-bit prefix, from the exclusive
// scan of its low-digit counts in LDS.
template <int THREADS>
__device__ __forceinline__ void emit_run(uint32_t* __restrict__ out, uint32_t prefix, uint32_t from,
                                         uint32_t to, const uint32_t* s_start) {
  for (uint32_t p = from + threadIdx.x; p < to; p += THREADS) {
    uint32_t v = 0;  // the last digit that starts at or before p
#pragma unroll
    for (uint32_t step = kRadix / 2; step; step >>= 1)
      if (s_start[v + step] <= p) v += step;
    out[p] = prefix | v;
  }
}

// The exclusive scan of 1024 counts into s_start.
template <int THREADS>
__device__ __forceinline__ void scan_counts(const uint32_t* counts, uint32_t* s_start,
                                            uint32_t* s_tmp) {
  constexpr int PER = kRadix / THREADS;
  const int tid = threadIdx.x;
  uint32_t c[PER];
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    c[j] = counts[tid * PER + j];
    sum += c[j];
  }
  uint32_t total;
  uint32_t run = block_excl_scan<THREADS>(sum, s_tmp, &total);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    s_start[tid * PER + j] = run;
    run += c[j];
  }
  __syncthreads();
}

// ... and the windows of the result, sorted from `in` into `out`.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void msd_l2_window_kernel(const uint32_t* __restrict__ in,
                                                            uint32_t* __restrict__ out,
                                                            MsdLevel2 l2,
                                                            const uint32_t* __restrict__ ctrl) {
  constexpr int WAVES = 8, KPT = 24, THREADS = 512;
  constexpr uint32_t CAP = THREADS * KPT;
  __shared__ uint32_t s_start[kRadix];
  __shared__ uint32_t s_tmp[WAVES];
  __shared__ uint32_t s_rank;
  const int32_t n_tiles = static_cast<int32_t>(ctrl[kCtrlMsdTiles]);
  if (n_tiles == 0 || stopped_any(ctrl)) return;
  const int tid = threadIdx.x;
  const int32_t t = blockIdx.x;
  if (t >= n_tiles) return;
  const int2 ref = l2.tiles[t];
  const int4 big = l2.big[ref.x];
  const uint32_t len = static_cast<uint32_t>(big.y);
  const uint32_t wlo = static_cast<uint32_t>(ref.y) * kL2Tile;
  const uint32_t whi = min(wlo + kL2Tile, len);
  const uint32_t top = static_cast<uint32_t>(big.z) << 20;
  const uint32_t* src = in + big.x;
  uint32_t* dst = out + big.x;
  uint32_t cnt[kRadix / THREADS];
  const Window w = find_window<THREADS>(l2.hist + static_cast<int64_t>(ref.x) * kRadix, -1, wlo,
                                        whi, cnt);
  // A shared run's part of this window, from the counts of its low bits.
  const auto shared_run = [&](uint32_t digit, uint32_t start, uint32_t from, uint32_t to) {
    __syncthreads();
    if (tid == 0) s_rank = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadix / THREADS; ++j)
      if (cnt[j] > kShare && static_cast<uint32_t>(tid * (kRadix / THREADS) + j) < digit)
        atomicAdd(&s_rank, 1u);
    __syncthreads();
    const uint32_t slot = static_cast<uint32_t>(big.w) + s_rank;
    if (slot >= static_cast<uint32_t>(l2.max_slots)) return;  // (never: sized for any keys)
    scan_counts<THREADS>(l2.hist3 + static_cast<int64_t>(slot) * kRadix, s_start, s_tmp);
    emit_run<THREADS>(dst + start, top | (digit << 10), from - start, to - start, s_start);
    __syncthreads();
  };
  if (w.reaches && w.cont_end - w.cont_start > kShare && w.cont_end <= len)
    shared_run(w.cont, w.cont_start, wlo, min(whi, w.cont_end));
  if (w.any && w.b <= len) {
    if (w.b - w.a <= CAP) {
      lds_bucket_sort<WAVES, KPT, 12, 8>(src + w.a, dst + w.a, static_cast<int32_t>(w.b - w.a),
                                         top | (w.first << 10),
                                         span_bits(w.last - w.first + 1u, 10));
      return;
    }
    if (w.c0 > w.a)
      lds_bucket_sort<WAVES, KPT, 12, 8>(src + w.a, dst + w.a, static_cast<int32_t>(w.c0 - w.a),
                                         top | (w.first << 10), span_bits(w.last - w.first, 10));
    const uint32_t n = w.b - w.c0;
    if (n <= CAP) {
      lds_bucket_sort<WAVES, KPT, 12, 8>(src + w.c0, dst + w.c0, static_cast<int32_t>(n),
                                         top | (w.last << 10), 10);
    } else {
      if (n > kShare) {
        shared_run(w.last, w.c0, w.c0, min(whi, w.b));
      } else {
        __shared__ uint32_t s_count[kRadix];
        __syncthreads();
        for (int k = tid; k < kRadix; k += THREADS) s_count[k] = 0;
        __syncthreads();
        for (uint32_t p = tid; p < n; p += THREADS) atomicAdd(&s_count[src[w.c0 + p] & 1023u], 1u);
        __syncthreads();
        scan_counts<THREADS>(s_count, s_start, s_tmp);
        emit_run<THREADS>(dst + w.c0, top | (w.last << 10), 0, n, s_start);
      }
    }
  }
}

}  // namespace

void launch_msd_scatter(const uint32_t* in, uint32_t* out, const SegView& sv,
                        const int32_t* tile_start, int32_t total_tiles, const uint32_t* hist,
                        uint32_t* cursor, const uint32_t* ctrl, const TuneTable& tt,
                        hipStream_t s) {
  if (total_tiles <= 0) return;
  // (the top digit's counts are slot 2 of each cloud's 10-bit histograms)
  const uint32_t* top = hist + 2 * kRadix;
  if (tt.sort10_kpt == 16)
    cursor_scatter_kernel<1024, 16, TopDigit10><<<total_tiles, 1024, 0, s>>>(
        in, out, sv, tile_start, nullptr, top, hist_stride(10), cursor, ctrl, TopDigit10{});
  else
    cursor_scatter_kernel<1024, 8, TopDigit10><<<total_tiles, 1024, 0, s>>>(
        in, out, sv, tile_start, nullptr, top, hist_stride(10), cursor, ctrl, TopDigit10{});
}

void launch_msd_windows(uint32_t* keys, const SegView& sv, const int32_t* tile_start,
                        int32_t total_tiles, int64_t max_seg, const uint32_t* hist,
                        const MsdLevel2& l2, uint32_t* ctrl, hipStream_t s) {
  if (total_tiles <= 0) return;
  // (four waves a workgroup: the windows of small segments)
  if (msd_small(max_seg))
    msd_window_kernel<4, 16, 10, 12><<<total_tiles, 256, 0, s>>>(keys, sv, tile_start, hist, l2,
                                                             ctrl);
  else
    msd_window_kernel<8, 24, 9, 13><<<total_tiles, 512, 0, s>>>(keys, sv, tile_start, hist, l2,
                                                            ctrl);
}

void launch_msd_level2(uint32_t* keys, uint32_t* other, const MsdLevel2& l2, int64_t n,
                       int64_t max_seg, const uint32_t* ctrl, hipStream_t s) {
  // Tiles that this build can list; the room may be that of a longer one before it
  // (20,000 points after a build of 30M: 70 us by the room, 60 as before it).
  MsdLevel2 need{};
  msd_level2_caps(n, max_seg, &need);
  const int32_t tiles = std::min(need.max_tiles, l2.max_tiles);
  // Counting takes a grid that fills the chip once, whose workgroups take every
  // grid-th tile; the scatter and the LDS sorts one tile each (in a loop the
  // compiler keeps a tile's addresses, and one scatter shares a CU instead of two:
  // 2^24 clustered points 457 -> 446 us).
  const uint32_t grid = static_cast<uint32_t>(std::max(1, std::min(tiles, 768)));
  msd_l2_hist_kernel<<<grid, 512, 0, s>>>(keys, l2, ctrl);
  msd_l2_scatter_kernel<<<static_cast<uint32_t>(tiles), 1024, 0, s>>>(keys, other, l2, ctrl);
  msd_l2_window_kernel<<<static_cast<uint32_t>(tiles), 512, 0, s>>>(other, keys, l2, ctrl);
}

}  // namespace ocp
