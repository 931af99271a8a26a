// Stage 4: Karras binary radix tree over the sorted unique codes, one
// thread per node, exactly the per-node function of
// kernels/04_radix_tree.cpp:47-120 (kernels/cuda/04_radix_tree.cu:33-113):
// direction from the two neighbours, exponential then binary search for
// the far end j, common-prefix length delta(i, j) = clz(a ^ b) - 1, binary
// search for the split gamma, leaf flags, parent links of internal
// children. clz runs on v_ffbh_u32 with clz(0) := 32.
//
// Parents without a race. The reference writes parent[] from every node;
// run sequentially the last writer wins. Nodes i >= 1 compute the standard
// Karras ranges over all U keys, so every internal node except the true
// root's children has exactly one writer among them. Node 0 is the
// quirk root: the reference gives it the range [0, n-1] instead of [0, n]
// (04_radix_tree.cpp:63-65), and it writes first, so whatever it writes is
// either overwritten by a node i >= 1 or lands on an entry nobody else
// writes, which the true root would own. Thread 0 therefore computes the
// true root split and stores 0 into parent[0] and into the parent entries
// of the true root's internal children; nodes i >= 1 store plainly. The
// result equals the sequential reference on zeroed memory without atomics
// or a zero-fill pass.
//
// Two kernels. radix_tree_kernel evaluates the reference's searches as they
// stand, for any sorted codes a caller passes (repeated ones and codes with
// bit 31 set included): the per-stage entry. radix_pairs_kernel is the fused
// build's, whose codes are always strictly increasing 30-bit keys.
#include "pair_rows.hpp"

namespace ocp {
namespace {

__device__ __forceinline__ int32_t log2_ceil(uint32_t x) {
  if (x == 0) return 0;
  const int32_t lo = 31 - static_cast<int32_t>(clz32(x));
  return lo + ((1u << lo) < x);
}

// Codes of a segment, served from an LDS window [lo, lo + n) when the
// index falls inside it. Most searches of a node stay close to the node.
struct Codes {
  const uint32_t* g;
  lds_ptr<const uint32_t> w;
  int32_t lo;
  int32_t n;
  __device__ __forceinline__ uint32_t operator[](int32_t q) const {
    return static_cast<uint32_t>(q - lo) < static_cast<uint32_t>(n) ? w[q - lo] : g[q];
  }
  // For an index known to lie in the window: no fallback branch.
  __device__ __forceinline__ uint32_t local(int32_t q) const { return w[q - lo]; }
};

// delta(code_i, c) > dl as one subtraction and compare, for a fixed dl in
// [0, 30]. With x = code_i ^ c: x == 0 gives delta 31 and x >= 2^31 gives
// delta 255 (clz 0, minus one, as a byte), both above dl; otherwise delta =
// clz(x) - 1 > dl exactly when x < 2^(30 - dl). So the predicate holds for
// x < lim or x >= 2^31, i.e. for x - lim >= 2^31 - lim (unsigned).
struct Above {
  uint32_t ci;
  uint32_t lim;
  uint32_t thr;
  __device__ __forceinline__ Above(uint32_t code_i, uint32_t dl)
      : ci(code_i), lim(1u << (30u - dl)), thr(0x80000000u - (1u << (30u - dl))) {}
  __device__ __forceinline__ bool operator()(uint32_t c) const { return ((c ^ ci) - lim) >= thr; }
};

#ifndef OCP_RADIX_HALO
#define OCP_RADIX_HALO 1024
#endif
// Codes staged on either side of a tile. 10M uniform keys: 128 -> 175 us,
// 256 -> 141 us, 512 -> 131 us (the neighbours' halos mostly hit in L2);
// with the wave path for wide nodes, 512 -> 110 us, 1024 -> 105 us,
// 2048 -> 109 us (2^24 clustered keys: 171, 160, 169 us).
constexpr int kHalo = OCP_RADIX_HALO;
// Nodes whose exponential search is still running at this length are
// finished by a whole wave; the rest stay inside the LDS window.
constexpr int32_t kLocalMax = kHalo / 2;
constexpr int kLocalLog = __builtin_ctz(kLocalMax);
static_assert((kLocalMax & (kLocalMax - 1)) == 0 && kLocalLog >= 1 && kLocalLog < 31,
              "the local search bound is a power of two");

// Split search of 04_radix_tree.cpp:94-104 for node i with far end j. The
// reference's divisor runs over 2, 4, ..., 2^log2_ceil(l) and its step is
// ceil(l / divisor); with power-of-two divisors that is a shift, so no
// integer division is left on the device.
// Only called for local nodes (l < kLocalMax), whose probes stay in the window.
template <bool CHECK>
__device__ __forceinline__ int32_t split_search(const Codes& codes, const Above& above,
                                                int32_t i, int32_t d,
                                                int32_t l, int32_t n) {
  int32_t s = 0;
  const int32_t lg = log2_ceil(static_cast<uint32_t>(l));
  const int32_t s_cutoff = (d == -1) ? i - 1 : n - i - 1;
  // l < kLocalMax, so lg <= kLocalLog: a fixed number of guarded steps.
#pragma unroll
  for (int32_t k = 1; k <= kLocalLog; ++k) {
    const int32_t t = static_cast<int32_t>((static_cast<uint32_t>(l) + (1u << k) - 1u) >> k);
    const int32_t st = s + t;
    const bool probe = k <= lg && (!CHECK || st <= s_cutoff);
    if (probe && above(codes.local(probe ? i + st * d : i))) s = st;
  }
  return i + s * d + min(d, 0);
}

// Wide nodes. All three searches of a node look for the largest x with a
// predicate that is monotone in x (codes are sorted, so the common prefix
// with code i only shrinks away from i): the reference's exponential search
// stops at the first power of two that fails, its binary searches return
// the largest x below their bound that holds (for the length: x < l_max and
// x <= l_cutoff; for the split: x <= min(l - 1, s_cutoff), the predicate
// failing at l). A whole wave evaluates 64 candidates per round trip
// instead of one, so a node spanning 2^k keys costs about k/6 dependent
// loads instead of 3k.
template <class Pred>
__device__ __forceinline__ int32_t wave_max_true(int32_t lo, int32_t hi, Pred pred) {
  // largest x in [lo, hi) with pred(x); pred(lo) holds.
  const int32_t lane = static_cast<int32_t>(lane_id());
  while (hi - lo > 1) {
    const int32_t step = (hi - lo + 63) >> 6;
    const int32_t x = lo + step * (lane + 1);
    const bool ok = x < hi && pred(x);
    const int32_t c = __popcll(__ballot(ok));
    const int32_t nlo = lo + step * c;
    hi = min(hi, lo + step * (c + 1));
    lo = nlo;
  }
  return lo;
}

struct NodeOut {
  uint32_t delta_node;
  int32_t gamma;
  int32_t j;
};

__device__ __forceinline__ NodeOut wave_node(const Codes& codes, int32_t i, int32_t n) {
  const int32_t lane = static_cast<int32_t>(lane_id());
  const uint32_t code_i = codes[i];
  int32_t d, l;
  if (i == 0) {
    d = 1;
    l = n - 1;
  } else {
    const int32_t diff = static_cast<int32_t>(delta(code_i, codes[i + 1])) -
                         static_cast<int32_t>(delta(code_i, codes[i - 1]));
    d = (diff > 0) - (diff < 0);
    const uint32_t delta_min = delta(code_i, codes[i - d]);
    // exponential search: lane k tests l_max = 2^k, k = 1..30
    bool ok = false;
    if (lane >= 1 && lane <= 30) {
      const int64_t q = static_cast<int64_t>(i) + (int64_t(1) << lane) * d;
      ok = q >= 0 && q <= n && delta(code_i, codes[static_cast<int32_t>(q)]) > delta_min;
    }
    const int32_t c = __popcll(__ballot(ok));
    const int32_t l_max = 1 << (c + 1);
    const int32_t l_cutoff = (d == -1) ? i : n - i;
    l = wave_max_true(0, min(l_max, l_cutoff + 1), [&](int32_t x) {
      return delta(code_i, codes[i + x * d]) > delta_min;
    });
  }
  NodeOut o;
  o.j = i + l * d;
  o.delta_node = delta(code_i, codes[o.j]);
  const int32_t s_cutoff = (d == -1) ? i - 1 : n - i - 1;
  const int32_t s = l <= 0 ? 0 : wave_max_true(0, min(l - 1, s_cutoff) + 1, [&](int32_t x) {
    return delta(code_i, codes[i + x * d]) > o.delta_node;
  });
  o.gamma = i + s * d + min(d, 0);
  return o;
}


// A node whose searches stay within kLocalMax of it, read from the LDS
// window without the window test (the window spans kHalo >= kLocalMax + 2
// around the tile). Returns false, emitting nothing, for a node the wave
// path must finish: a far end beyond kLocalMax, or a threshold of 31 or
// above (repeated codes, codes with bit 31 set), for which the wave path
// evaluates delta itself. CHECK: bound the probes by [0, n] and the
// reference's length and split cutoffs (tiles near either end).
template <bool CHECK, class Emit>
__device__ __forceinline__ bool local_node(const Codes& codes, int32_t i, int32_t n,
                                           Emit& emit) {
  const uint32_t code_i = codes.local(i);
  const uint32_t dn = delta(code_i, codes.local(i + 1));
  const uint32_t dp = delta(code_i, codes.local(i - 1));
  const int32_t diff = static_cast<int32_t>(dn) - static_cast<int32_t>(dp);
  const int32_t d = (diff > 0) - (diff < 0);
  // delta(code_i, codes[i - d]); d == 0 (equal neighbours, repeated codes
  // only) compares code i with itself: 31.
  const uint32_t delta_min = d > 0 ? dp : (d < 0 ? dn : 31u);
  if (delta_min >= 31u) return false;
  const Above above_min(code_i, delta_min);
  // Exponential search for an upper bound l_max (a power of two), then
  // binary search of the length: t = l_max / 2, l_max / 4, ..., 1. The
  // reference probes 2, 4, 8, ... until one fails; here the probes up to
  // kLocalMax are read at once and l_max = 2^(leading passes + 1).
  uint32_t pass = 0;
#pragma unroll
  for (int k = 1; k <= kLocalLog; ++k) {
    const int32_t q = i + (1 << k) * d;
    const bool in = !CHECK || (q >= 0 && q <= n);
    const uint32_t cq = codes.local(in ? q : i);
    pass |= static_cast<uint32_t>(in && above_min(cq)) << (k - 1);
  }
  const int32_t l_max = 2 << __builtin_ctz(~pass);
  if (l_max > kLocalMax) return false;
  const int32_t l_cutoff = (d == -1) ? i : n - i;
  int32_t l = 0;
#pragma unroll
  for (int k = 1; k <= kLocalLog; ++k) {  // t = l_max / 2, l_max / 4, ..., 1
    const int32_t t = l_max >> k;
    const bool probe = t >= 1 && (!CHECK || l + t <= l_cutoff);
    if (probe && above_min(codes.local(probe ? i + (l + t) * d : i))) l += t;
  }
  const int32_t j = i + l * d;
  const uint32_t delta_node = delta(code_i, codes.local(j));
  if (delta_node >= 31u) return false;
  emit(i, delta_node, split_search<CHECK>(codes, Above(code_i, delta_node), i, d, l, n), j);
  return true;
}

__global__ __launch_bounds__(256) void radix_tree_kernel(
    const uint32_t* __restrict__ codes_g, uint8_t* __restrict__ prefix_n,
    uint8_t* __restrict__ hl, uint8_t* __restrict__ hr, int32_t* __restrict__ lc,
    int32_t* __restrict__ parent, int32_t n, const uint32_t* __restrict__ ctrl) {
  static_assert(kLocalMax <= kHalo / 2 + 1, "local searches must stay in the window");
  __shared__ uint32_t s_codes[kNodeTile + 2 * kHalo];
  __shared__ int32_t s_wide[kNodeTile];
  __shared__ uint32_t s_nwide;
  const int32_t i0 = xcd_tile(blockIdx.x, gridDim.x) * kNodeTile;
  // After a lookback time-out the unique keys are not valid input.
  if (i0 >= n || (ctrl && stopped_any(ctrl))) return;
  if (threadIdx.x == 0) s_nwide = 0;
  // Stage codes [i0 - halo, i0 + kNodeTile + halo) of the n+1 codes.
  const int32_t lo = max(0, i0 - kHalo);
  const int32_t hi = min(n + 1, i0 + kNodeTile + kHalo);
  {
    // every load of the window in flight at once
    constexpr int kRows = (kNodeTile + 2 * kHalo + 255) / 256;
    uint32_t rc[kRows];
    const uint32_t* src = codes_g + lo + static_cast<int32_t>(threadIdx.x);
    if (hi - lo == kRows * 256) {  // a full window: no per-load guard
#pragma unroll
      for (int k = 0; k < kRows; ++k) rc[k] = src[k * 256];
    } else {
#pragma unroll
      for (int k = 0; k < kRows; ++k)
        if (lo + static_cast<int32_t>(threadIdx.x) + k * 256 < hi) rc[k] = src[k * 256];
    }
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
      const int32_t q = lo + static_cast<int32_t>(threadIdx.x) + k * 256;
      if (q < hi) s_codes[q - lo] = rc[k];
    }
  }
  __syncthreads();
  const Codes codes{codes_g, as_lds<const uint32_t>(s_codes), lo, hi - lo};

  auto emit = [&](int32_t node, uint32_t delta_node, int32_t gamma, int32_t j) {
    const bool leaf_l = min(node, j) == gamma;
    const bool leaf_r = max(node, j) == gamma + 1;
    prefix_n[node] = static_cast<uint8_t>(delta_node);
    hl[node] = leaf_l;
    hr[node] = leaf_r;
    lc[node] = gamma;
    if (node > 0) {
      if (!leaf_l) parent[gamma] = node;
      if (!leaf_r) parent[gamma + 1] = node;
    }
  };

  // A tile at least 2 * kLocalMax away from both ends of [0, n]: every
  // probe of a local node (within kLocalMax + 2 of i) is inside [0, n] and
  // below the length and split cutoffs, so those checks are skipped.
  const bool interior = i0 >= 2 * kLocalMax && i0 + kNodeTile + 2 * kLocalMax <= n;
  for (int32_t k = 0; k < kNodeTile / 256; ++k) {
  const int32_t i = i0 + k * 256 + static_cast<int32_t>(threadIdx.x);
  bool wide = false;
  if (i < n) {
    if (i == 0) {
      wide = true;
    } else {
      wide = interior ? !local_node<false>(codes, i, n, emit)
                      : !local_node<true>(codes, i, n, emit);
    }
  }
  const uint64_t bal = __ballot(wide);
  if (bal) {
    uint32_t base = 0;
    if (lane_id() == 0) base = atomicAdd(&s_nwide, static_cast<uint32_t>(__popcll(bal)));
    base = __shfl(base, 0, 64);
    if (wide) s_wide[base + __popcll(bal & lanemask_lt())] = i;
  }
  }
  __syncthreads();
  const uint32_t nw = s_nwide;
  for (uint32_t q = wave_id(); q < nw; q += 4) {
    const int32_t node = s_wide[q];
    const NodeOut o = wave_node(codes, node, n);
    if (lane_id() == 0) emit(node, o.delta_node, o.gamma, o.j);
    if (node == 0) {
      // The true root spans [0, n]: its internal children have no other
      // writer, and sequentially they end up holding node 0. Its split is
      // the largest s <= n - 1 with delta(c0, codes[s]) > delta(c0, codes[n]).
      const uint32_t c0 = codes[0];
      const uint32_t dn = delta(c0, codes[n]);
      const int32_t g0 = wave_max_true(0, n, [&](int32_t q) { return delta(c0, codes[q]) > dn; });
      if (lane_id() == 0) {
        parent[0] = 0;
        if (g0 != 0 && g0 < n) parent[g0] = 0;
        if (g0 + 1 != n && g0 + 1 < n) parent[g0 + 1] = 0;
      }
    }
  }
}

// ---------------------------------------------------------------- fused build
// The fused build's keys are strictly increasing 30-bit codes, and there the
// tree is the Cartesian tree of the adjacent pairs: with b_k = clz(c_k ^
// c_(k+1)) (the pair's common prefix, plus two), the internal node that splits
// between keys k and k+1 spans the pairs around k up to the nearest smaller b
// on either side, L < k < R, so the keys L+1 .. R (two equal values always
// have a smaller one between them). Its parent is the pair at whichever end
// holds the larger b; the reference's index for the node is L+1 when that is
// L (a right child starts its range) and R otherwise. Everything the stage
// writes follows: prefix_n = b_k - 1, left_child = k, the leaf flags from
// L+1 == k and R == k+1, the children's parents (nodes k and k+1), and also
// the edge count of stage 5 (kernels/05_edge_count.cpp:3-16), for the parent's
// prefix length is max(b_L, b_R) - 1.
//
// The pairs' b values of a tile and its halo lie in LDS as bytes, with the
// minima of 16 and of 256 of them: three levels of 16-byte rows. One row is
// compared with b_k by four byte-wise subtractions whose top bits four dot
// products collect into a 16-bit mask. The masks of the pair's own row and of the
// one nearer to it give the nearest smaller value on both sides of five pairs in
// six; the others are listed and searched a full wave at a time: their own row,
// else the row of row minima names the row to look into, else that of the
// 256-pair minima. Values outside the
// segment are 0, below any pair's. An end beyond the window is searched by
// the wave in the codes themselves, 64 candidates a round trip.
//
// Results leave by node index: the records of a tile's own indices through
// LDS and then as 4-node stores; the others, whose node index lies in another
// tile, one by one. Every index has one pair, so no entry is stored twice.
//
// Node 0 is the reference's short root (see the top of this file): its record
// comes from its own search, the true root's pair only links its children, and
// those count their edges from node 0's prefix length.
//
// What bounds it: vector instructions and stores. 10M uniform points take 55 us
// (the 190 MB it moves 37 at the rate of a large copy), 2^24 clustered ones 31;
// searching every pair at all three levels, because some lane of a wave needs
// each, 66 and 37; the searches by code of the kernel above 99 us, with an edge
// scan of 33 us that formed the counts it now reads (22). The halo is 512 pairs
// for tiles of 2048 and 256 for those of 512 (2^20 points 17.3 us with 512, 16.8).
// The end of the run of keys around key `from` whose xor with code c is below
// lim, at least `reach` keys away on the side of d (+1, -1), in [0, m].
__device__ __forceinline__ int32_t wave_run_end(const uint32_t* __restrict__ codes, uint32_t c,
                                                uint32_t lim, int32_t from, int32_t d, int32_t m) {
  const int32_t room = d > 0 ? m - from : from;  // steps that stay in [0, m]
  const auto in_run = [&](int32_t x) { return (codes[from + x * d] ^ c) < lim; };
  const int32_t lane = static_cast<int32_t>(lane_id());
  bool ok = false;
  if (lane < 30) {
    const int32_t x = 1 << lane;
    ok = x <= room && in_run(x);
  }
  const int32_t n = __popcll(__ballot(ok));
  return from + d * wave_max_true(n ? 1 << (n - 1) : 0, min(1 << n, room + 1), in_run);
}

template <int T, int HALO>
__global__ __launch_bounds__(256) void radix_pairs_kernel(
    const uint32_t* __restrict__ codes_all, uint8_t* __restrict__ prefix_all,
    uint8_t* __restrict__ hl_all, uint8_t* __restrict__ hr_all, int32_t* __restrict__ lc_all,
    int32_t* __restrict__ par_all, int32_t* __restrict__ edge_all, SegView sv,
    const int32_t* __restrict__ tile_start, const int32_t* __restrict__ n_unique,
    const uint32_t* __restrict__ ctrl) {
  constexpr int W = T + 2 * HALO;
  constexpr int ROWS = W / 256;
  static_assert(T % 512 == 0 && T <= 2048 && W % 256 == 0 && W <= 4096, "three levels of 16");
  __shared__ v4u s_b[W / 16];    // b of the window's pairs, a byte each
  __shared__ v4u s_b16[16];      // minima of 16
  __shared__ v4u s_b256;         // minima of 256
  __shared__ uint32_t s_rec[T];  // records of the tile's node indices
  __shared__ int32_t s_par[T];
  __shared__ uint16_t s_list[4][128];
  constexpr uint32_t kNone = 0xffffffffu;

  const TileRef r = find_tile(tile_start, sv.n_seg, xcd_tile(blockIdx.x, gridDim.x));
  const int32_t m = n_unique[r.seg] - 1;  // pairs 0 .. m-1 between keys 0 .. m
  const int32_t sb = seg_begin(sv, r.seg);
  const int32_t i0 = r.local * T;
  // After a lookback time-out the unique keys are not valid input.
  if (i0 >= m || stopped_any(ctrl)) return;
  const uint32_t* codes = codes_all + sb;
  uint8_t* prefix = prefix_all + sb;
  uint8_t* hl = hl_all + sb;
  uint8_t* hr = hr_all + sb;
  int32_t* lc = lc_all + sb;
  int32_t* par = par_all + sb;
  int32_t* edge = edge_all + sb;
  const int tid = threadIdx.x;
  const int32_t wb = i0 - HALO;
  const uint32_t code_0 = codes[0], code_m = codes[m], code_l = codes[m - 1];

  {
    // every load of the window in flight at once
    uint32_t a[ROWS], c[ROWS];
    if (wb >= 0 && wb + W <= m) {
      const uint32_t* src = codes + wb + tid;
#pragma unroll
      for (int k = 0; k < ROWS; ++k) {
        a[k] = src[k * 256];
        c[k] = src[k * 256 + 1];
      }
    } else {
#pragma unroll
      for (int k = 0; k < ROWS; ++k) {
        const int32_t g = wb + tid + k * 256;
        a[k] = 0u;
        c[k] = 0x80000000u;  // clz 0: outside the segment
        if (g >= 0 && g < m) {
          a[k] = codes[g];
          c[k] = codes[g + 1];
        }
      }
    }
    uint8_t* b = reinterpret_cast<uint8_t*>(s_b);
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
      b[tid + k * 256] = static_cast<uint8_t>(__clz(static_cast<int>(a[k] ^ c[k])));
    for (int k = tid; k < T; k += 256) {
      s_rec[k] = kNone;
      s_par[k] = -1;
    }
  }
  __syncthreads();
  reinterpret_cast<uint8_t*>(s_b16)[tid] =
      static_cast<uint8_t>(tid < W / 16 ? min16(s_b[tid]) : 31u);
  __syncthreads();
  if (tid < 16) reinterpret_cast<uint8_t*>(&s_b256)[tid] = static_cast<uint8_t>(min16(s_b16[tid]));
  __syncthreads();

  const uint32_t b_root = static_cast<uint32_t>(__clz(static_cast<int>(code_0 ^ code_m)));
  const uint32_t pn_0 = delta(code_0, code_l);  // node 0's prefix length
  const uint8_t* b8 = reinterpret_cast<const uint8_t*>(s_b);
  const v4u row256 = s_b256;

  // What a pair's two ends give.
  const auto emit = [&](int32_t p, uint32_t b, int32_t pl, int32_t pr, uint32_t b_l,
                        uint32_t b_r) {
    const int32_t g = i0 + p;
    const uint32_t b_up = max(b_l, b_r);
    const int32_t node = b_l >= b_r ? pl + 1 : pr;
    const bool leaf_l = pl + 1 == g;
    const bool leaf_r = pr == g + 1;
    const uint32_t pn = b - 1u;
    const int32_t e = static_cast<int32_t>(third(pn)) -
                      static_cast<int32_t>(third(b_up == b_root ? pn_0 : b_up - 1u));
    const uint32_t rec = static_cast<uint32_t>(p) | (pn << 11) | (leaf_l ? 1u << 16 : 0u) |
                         (leaf_r ? 1u << 17 : 0u) | (static_cast<uint32_t>(e + 16) << 18);
    const int32_t rel = node - i0;
    if (b_up == 0) {
      // the true root: node 0's record is written below
    } else if (static_cast<uint32_t>(rel) < static_cast<uint32_t>(T)) {
      s_rec[rel] = rec;
    } else {
      prefix[node] = static_cast<uint8_t>(pn);
      hl[node] = leaf_l;
      hr[node] = leaf_r;
      lc[node] = g;
      edge[node] = e;
    }
    if (!leaf_l) s_par[p] = node;
    if (!leaf_r) {
      if (p + 1 < T) s_par[p + 1] = node;
      else par[g + 1] = node;
    }
  };
  // Most ends lie within eight pairs: every pair is compared with the two rows
  // nearest to it; those for which that is not enough are listed.
  uint32_t listed = 0;
  uint16_t* list = s_list[wave_id()];
  const int32_t lane = static_cast<int32_t>(lane_id());
#pragma unroll 1
  for (int k = 0; k < T / 256; ++k) {
    {
      const int32_t p = k * 256 + tid;  // place in the tile
      const bool live = i0 + p < m;
      const uint32_t q = static_cast<uint32_t>(p + HALO);
      const uint32_t b = b8[q];
      const uint32_t key = __builtin_amdgcn_perm(0u, b + 127u, 0u);
      const uint32_t row = (q - 8u) >> 4;
      const uint32_t pos = q - row * 16u;
      const uint32_t hits = below16(s_b[row], key) | (below16(s_b[row + 1], key) << 16);
      const uint32_t to_r = hits & (0xfffffffeu << pos), to_l = hits & ((1u << pos) - 1u);
      const bool found = to_r != 0 && to_l != 0;
      if (live && found) {
        const int32_t end_r = static_cast<int32_t>(row * 16u) + __builtin_ctz(to_r);
        const int32_t end_l =
            static_cast<int32_t>(row * 16u) + 31 - __clz(static_cast<int>(to_l));
        emit(p, b, wb + end_l, wb + end_r, b8[end_l], b8[end_r]);
      }
      const uint64_t more = __ballot(live && !found);
      if ((more >> lane) & 1u)
        list[listed + static_cast<uint32_t>(__popcll(more & lanemask_lt()))] =
            static_cast<uint16_t>(p);
      listed += static_cast<uint32_t>(__popcll(more));
    }
    while (listed >= (k == T / 256 - 1 ? 1u : 64u)) {
      const uint32_t batch = min(listed, 64u);
      listed -= batch;
      const bool live = static_cast<uint32_t>(lane) < batch;
      const int32_t p = live ? list[listed + lane] : 0;
      const int32_t g = i0 + p;  // the pair
      const uint32_t q = static_cast<uint32_t>(p + HALO);
      const uint32_t b = b8[q];
      // (b + 127 in every byte; a dead lane looks for the first pair's, to no end)
      const uint32_t key = __builtin_amdgcn_perm(0u, b + 127u, 0u);
      const uint32_t row = q >> 4, grp = q >> 8;
      const uint32_t m0 = below16(s_b[row], key);
      const uint32_t m1 = below16(s_b16[grp], key);
      const uint32_t m2 = below16(row256, key);
      int32_t end_l = -2, end_r = -2;  // window positions of L and R, -2: not in the window
      uint32_t hit = m0 & (0xfffeu << (q & 15u)) & 0xffffu;
      uint32_t at = row;
      if (hit == 0) {
        uint32_t gg = grp;
        uint32_t rr = m1 & (0xfffeu << (row & 15u)) & 0xffffu;
        if (rr == 0) {
          const uint32_t g2 = m2 & (0xfffeu << grp) & 0xffffu;
          if (g2) {
            gg = static_cast<uint32_t>(__builtin_ctz(g2));
            rr = below16(s_b16[gg], key);
          }
        }
        if (rr) {
          at = gg * 16u + static_cast<uint32_t>(__builtin_ctz(rr));
          hit = below16(s_b[at], key);
        }
      }
      if (hit) end_r = static_cast<int32_t>(at * 16u + static_cast<uint32_t>(__builtin_ctz(hit)));
      hit = m0 & ((1u << (q & 15u)) - 1u);
      at = row;
      if (hit == 0) {
        uint32_t gg = grp;
        uint32_t rr = m1 & ((1u << (row & 15u)) - 1u);
        if (rr == 0) {
          const uint32_t g2 = m2 & ((1u << grp) - 1u);
          if (g2) {
            gg = 31u - static_cast<uint32_t>(__clz(static_cast<int>(g2)));
            rr = below16(s_b16[gg], key);
          }
        }
        if (rr) {
          at = gg * 16u + 31u - static_cast<uint32_t>(__clz(static_cast<int>(rr)));
          hit = below16(s_b[at], key);
        }
      }
      if (hit) end_l = static_cast<int32_t>(at * 16u + 31u - static_cast<uint32_t>(__clz(static_cast<int>(hit))));
      uint32_t b_l = end_l >= 0 ? b8[end_l] : 0u;
      uint32_t b_r = end_r >= 0 ? b8[end_r] : 0u;
      int32_t pl = wb + end_l, pr = wb + end_r;  // the pairs L and R
      // Ends beyond the window, one at a time by the whole wave. The window's
      // last key (first key) is then still in the run.
      for (uint64_t far = __ballot(live && end_r < 0); far; far &= far - 1) {
        const int src = __builtin_ctzll(far);
        const int32_t gs = __builtin_amdgcn_readlane(g, src);
        const uint32_t lim = 1u << (32u - __builtin_amdgcn_readlane(b, src));
        const int32_t j = wave_run_end(codes, codes[gs + 1], lim, wb + W, 1, m);
        const uint32_t bj = j < m ? clz32(codes[j] ^ codes[j + 1]) : 0u;
        if (static_cast<int>(lane_id()) == src) {
          pr = j;
          b_r = bj;
        }
      }
      for (uint64_t far = __ballot(live && end_l < 0); far; far &= far - 1) {
        const int src = __builtin_ctzll(far);
        const int32_t gs = __builtin_amdgcn_readlane(g, src);
        const uint32_t lim = 1u << (32u - __builtin_amdgcn_readlane(b, src));
        const int32_t j = wave_run_end(codes, codes[gs], lim, wb, -1, m);
        const uint32_t bj = j > 0 ? clz32(codes[j - 1] ^ codes[j]) : 0u;
        if (static_cast<int>(lane_id()) == src) {
          pl = j - 1;
          b_l = bj;
        }
      }
      if (live) emit(p, b, pl, pr, b_l, b_r);
    }
  }
  __syncthreads();

  for (int v = tid; v < T / 4; v += 256) {
    const v4u x = reinterpret_cast<const v4u*>(s_rec)[v];
    const int32_t n0 = i0 + 4 * v;
    const auto bytes = [&](uint32_t shift, uint32_t mask) {
      return ((x.x >> shift) & mask) | (((x.y >> shift) & mask) << 8) |
             (((x.z >> shift) & mask) << 16) | (((x.w >> shift) & mask) << 24);
    };
    if (max(max(x.x, x.y), max(x.z, x.w)) != kNone) {
      const uint32_t w_pn = bytes(11, 31u), w_hl = bytes(16, 1u), w_hr = bytes(17, 1u);
      const v4u w_lc = (x & 2047u) + static_cast<uint32_t>(i0);
      const v4u w_e = ((x >> 18) & 63u) - 16u;
      __builtin_memcpy(prefix + n0, &w_pn, 4);
      __builtin_memcpy(hl + n0, &w_hl, 4);
      __builtin_memcpy(hr + n0, &w_hr, 4);
      __builtin_memcpy(lc + n0, &w_lc, 16);
      __builtin_memcpy(edge + n0, &w_e, 16);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t y = x[u];
        if (y == kNone) continue;
        prefix[n0 + u] = static_cast<uint8_t>((y >> 11) & 31u);
        hl[n0 + u] = static_cast<uint8_t>((y >> 16) & 1u);
        hr[n0 + u] = static_cast<uint8_t>((y >> 17) & 1u);
        lc[n0 + u] = i0 + static_cast<int32_t>(y & 2047u);
        edge[n0 + u] = static_cast<int32_t>((y >> 18) & 63u) - 16;
      }
    }
    const v4i w_par = reinterpret_cast<const v4i*>(s_par)[v];
    if (min(min(w_par.x, w_par.y), min(w_par.z, w_par.w)) >= 0) {
      __builtin_memcpy(par + n0, &w_par, 16);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (w_par[u] >= 0) par[n0 + u] = w_par[u];
    }
  }
  if (i0 == 0 && wave_id() == 0) {
    // Node 0: the range [0, m - 1] and its split (04_radix_tree.cpp:63-65,
    // 94-104): the largest s < m - 1 with a longer common prefix than pn_0.
    const int32_t s = m < 2 ? 0 : wave_max_true(0, m - 1, [&](int32_t x) {
      return delta(code_0, codes[x]) > pn_0;
    });
    if (lane_id() == 0) {
      prefix[0] = static_cast<uint8_t>(pn_0);
      hl[0] = s == 0;
      hr[0] = s + 1 == m - 1;
      lc[0] = s;
      par[0] = 0;
      edge[0] = 0;
    }
  }
}

}  // namespace

void launch_radix_tree(const uint32_t* codes, uint8_t* prefix_n, uint8_t* has_leaf_left,
                       uint8_t* has_leaf_right, int32_t* left_child, int32_t* parent, int32_t n,
                       const uint32_t* ctrl, hipStream_t s) {
  if (n <= 0) return;
  static_assert(kNodeTile % 256 == 0, "whole node rows per thread");
  radix_tree_kernel<<<(n + kNodeTile - 1) / kNodeTile, 256, 0, s>>>(
      codes, prefix_n, has_leaf_left, has_leaf_right, left_child, parent, n, ctrl);
}

void launch_radix_pairs(const uint32_t* codes, uint8_t* prefix_n, uint8_t* has_leaf_left,
                        uint8_t* has_leaf_right, int32_t* left_child, int32_t* parent,
                        int32_t* edge, const SegView& sv, const int32_t* tile_start,
                        int32_t total_tiles, int tile, const int32_t* n_unique,
                        const uint32_t* ctrl, hipStream_t s) {
  if (total_tiles <= 0) return;
  const auto go = [&](auto kernel) {
    kernel<<<total_tiles, 256, 0, s>>>(codes, prefix_n, has_leaf_left, has_leaf_right, left_child,
                                       parent, edge, sv, tile_start, n_unique, ctrl);
  };
  if (tile == 2048) go(radix_pairs_kernel<2048, 512>);
  else go(radix_pairs_kernel<512, 256>);
}

}  // namespace ocp
