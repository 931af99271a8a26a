// Octree output formats and a structural validator, on the device.
//
// Validator (in the role of checkTree, apps/cpu_demo/main.cpp:13-35): the
// reference's offsets are an inclusive scan used as first slots
// (kernels/06_partial_sum.cpp:3-15, include/shared/oct.h:24-90), so chains
// overlap and overwrite each other's geometry and child-in-octant does not
// hold in its own output. What holds whatever the write order, and is counted
// here per kind of violation:
//  - the written slots are slot 0 and the chain ranges [P[i], P[i] + e[i]) of
//    the radix-tree nodes i >= 1, and every chain ends inside its segment;
//    every other slot is all zero;
//  - a written slot has w = 1, a cell size range / 2^k (k = 0..11) and a
//    corner on the grid of octree level root_level + k (morton.h:45-80 with
//    oct.h:56-57, 87-88);
//  - child_leaf_mask is 0 (SetLeaf clears bits of a zeroed word, oct.h:17-21);
//  - the root slot holds the root corner and cell size = range.
// The node-mask links whose child slot lies inside the parent's octant are
// counted as information only.
//
// Compact nodes: a 12-byte header per slot - the corner as the Morton prefix
// whose decode it is, the octree level and the depth below the root (the
// cell size is range / 2^depth), the two masks, a bit per nonzero child and
// the index of its first stored child - and the nonzero children in one
// array. Expanding gives back the 60-byte nodes bit for bit. A slot that no
// chain writes has level byte 0xff.
#include "ocp_internal.hpp"

namespace ocp {
namespace {

constexpr int kFmtThreads = 256;
constexpr int kFmtGrid = 4096;

__device__ __forceinline__ uint32_t level_shift(int32_t level) {
  return level >= 10 ? 0u : static_cast<uint32_t>(kMortonBits - 3 * level);
}

// The segment holding global slot g: the last k with oct_start[k] <= g
// (empty segments before it share its start).
__device__ __forceinline__ int32_t seg_of_slot(int64_t g, const int32_t* oct_start,
                                               int32_t n_seg) {
  int32_t lo = 0, hi = n_seg;
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (oct_start[mid] <= g) lo = mid; else hi = mid;
  }
  return lo;
}

struct Boxes {
  const float* mn;  // per segment, or nullptr: mn1 / rg1
  const float* rg;
  float mn1, rg1;
  __device__ __forceinline__ float min_of(int32_t s) const { return mn ? mn[s] : mn1; }
  __device__ __forceinline__ float range_of(int32_t s) const { return rg ? rg[s] : rg1; }
};

// Depth k (0..11) with range / 2^k == cell bit for bit (the octree's own
// expression), or -1.
__device__ __forceinline__ int32_t depth_of(float cell, float rg) {
  for (int32_t k = 0; k <= 11; ++k) {
    const uint32_t sh = static_cast<uint32_t>(k) & 31u;
    if (__float_as_uint(rg / static_cast<float>(static_cast<int32_t>(1u << sh))) ==
        __float_as_uint(cell))
      return k;
  }
  return -1;
}

// The axis value q in [0, 1024), a multiple of 2^(10 - level), whose decode
// is c bit for bit, or -1. q is near (c - min) / range * 1024; the decode
// itself decides.
__device__ __forceinline__ int32_t axis_value(float c, int axis, int32_t level, float mn,
                                              float rg) {
  const double qd = (static_cast<double>(c) - mn) / rg * 1024.0;
  if (!(qd > -4.0 && qd < 1028.0)) return -1;
  const int32_t q0 = static_cast<int32_t>(floor(qd));
  const uint32_t grid = (1u << (level_shift(level) / 3u)) - 1u;
  for (int32_t d = -1; d <= 2; ++d) {
    const int32_t q = q0 + d;
    if (q < 0 || q > 1023 || (static_cast<uint32_t>(q) & grid)) continue;
    const uint32_t code = split_by_3(static_cast<uint32_t>(q)) << axis;
    if (__float_as_uint(decode_axis(code, axis, mn, rg)) == __float_as_uint(c)) return q;
  }
  return -1;
}

// The Morton prefix of `level` whose decode is the corner, or ~0u.
__device__ __forceinline__ uint32_t prefix_of(const float* c, int32_t level, float mn, float rg) {
  uint32_t code = 0;
  for (int a = 0; a < 3; ++a) {
    const int32_t q = axis_value(c[a], a, level, mn, rg);
    if (q < 0) return ~0u;
    code |= split_by_3(static_cast<uint32_t>(q)) << a;
  }
  return code;
}

__device__ __forceinline__ bool any_word(const OctNode& nd) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(&nd);
  uint32_t o = 0;
#pragma unroll
  for (int q = 0; q < 15; ++q) o |= w[q];
  return o != 0;
}

// Root level (prefix_n[0] / 3, 0 below two keys) and first code per segment.
__global__ void seg_roots_kernel(const uint32_t* __restrict__ codes,
                                 const uint8_t* __restrict__ prefix_n,
                                 const int32_t* __restrict__ n_unique,
                                 const int32_t* __restrict__ seg_start, int32_t n_seg,
                                 int32_t* __restrict__ root_level, uint32_t* __restrict__ root_code) {
  const int32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_seg) return;
  const int32_t sb = seg_start ? seg_start[s] : 0;
  const int32_t u = n_unique[s];
  root_level[s] = u >= 2 ? prefix_n[sb] / 3 : 0;
  root_code[s] = u >= 1 ? codes[sb] : 0u;
}

enum Report : int {
  kRepSlots = 0, kRepWritten, kRepCoveredUnwritten, kRepWrittenUncovered, kRepChainPastEnd,
  kRepBadW, kRepBadCell, kRepOffGrid, kRepLeafMask, kRepBadRoot, kRepLinks,
  kRepLinksInOctant, kRepFields
};

__device__ __forceinline__ void add_report(unsigned long long* rep, int field, uint32_t v) {
  v = wave_sum(v);
  if (lane_id() == 0 && v) atomicAdd(&rep[field], static_cast<unsigned long long>(v));
}

// cov[slot] = 1 for every slot of a chain (cov zeroed beforehand; chains of
// one segment may overlap, all store the same value). Grid: x over radix-tree
// nodes, y over segments.
__global__ __launch_bounds__(kFmtThreads) void cover_kernel(
    const int32_t* __restrict__ edge, const int32_t* __restrict__ offs,
    const int32_t* __restrict__ n_unique, const int32_t* __restrict__ oct_start,
    const int32_t* __restrict__ seg_start, int32_t n_seg, uint8_t* __restrict__ cov,
    unsigned long long* __restrict__ rep) {
  uint32_t past = 0;
  for (int32_t seg = blockIdx.y; seg < n_seg; seg += gridDim.y) {
    const int32_t m = n_unique[seg] - 1;
    const int32_t sb = seg_start ? seg_start[seg] : 0;
    const int32_t nb = oct_start[seg];
    const int32_t k = oct_start[seg + 1] - nb;
    for (int32_t i = blockIdx.x * kFmtThreads + threadIdx.x + 1; i < m;
         i += gridDim.x * kFmtThreads) {
      const int32_t e = edge[sb + i];
      if (e <= 0) continue;
      const int32_t p = offs[sb + i];
      if (p < 0 || p > k - e) {
        ++past;
        continue;
      }
      for (int32_t j = 0; j < e; ++j) cov[nb + p + j] = 1;
    }
  }
  add_report(rep, kRepChainPastEnd, past);
}

__global__ __launch_bounds__(kFmtThreads) void validate_kernel(
    const OctNode* __restrict__ nodes, const uint8_t* __restrict__ cov,
    const int32_t* __restrict__ oct_start, int32_t n_seg, Boxes bx,
    const int32_t* __restrict__ root_level, const uint32_t* __restrict__ root_code,
    unsigned long long* __restrict__ rep) {
  uint32_t cnt[kRepFields] = {};
  const int64_t k_total = oct_start[n_seg];
  for (int64_t g = blockIdx.x * int64_t(kFmtThreads) + threadIdx.x; g < k_total;
       g += int64_t(gridDim.x) * kFmtThreads) {
    const int32_t seg = seg_of_slot(g, oct_start, n_seg);
    const int32_t base = oct_start[seg];
    const int32_t local = static_cast<int32_t>(g - base);
    const int32_t k = oct_start[seg + 1] - base;
    const OctNode nd = nodes[g];
    const bool written = any_word(nd);
    const bool covered = local == 0 || cov[g] != 0;
    ++cnt[kRepSlots];
    cnt[kRepWritten] += written;
    cnt[kRepCoveredUnwritten] += covered && !written;
    cnt[kRepWrittenUncovered] += written && !covered;
    if (!written) continue;
    const float mn = bx.min_of(seg), rg = bx.range_of(seg);
    const int32_t rl = root_level[seg];
    cnt[kRepBadW] += __float_as_uint(nd.corner[3]) != __float_as_uint(1.0f);
    cnt[kRepLeafMask] += nd.child_leaf_mask != 0;
    const int32_t depth = depth_of(nd.cell_size, rg);
    if (depth < 0) {
      ++cnt[kRepBadCell];
      continue;
    }
    const uint32_t pre = prefix_of(nd.corner, rl + depth, mn, rg);
    cnt[kRepOffGrid] += pre == ~0u;
    if (local == 0) {
      const uint32_t sh = level_shift(rl);
      const uint32_t c0 = (root_code[seg] >> sh) << sh;
      bool same = depth == 0;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        same &= __float_as_uint(decode_axis(c0, a, mn, rg)) == __float_as_uint(nd.corner[a]);
      cnt[kRepBadRoot] += !same;
    }
    const float h = nd.cell_size * 0.5f;
    for (int c = 0; c < 8; ++c) {
      if (!((nd.child_node_mask >> c) & 1)) continue;
      ++cnt[kRepLinks];
      const int32_t t = nd.children[c];
      if (t < 0 || t >= k) continue;
      const OctNode ch = nodes[base + t];
      const float lo0 = nd.corner[0] + ((c & 1) ? h : 0.0f);
      const float lo1 = nd.corner[1] + ((c & 2) ? h : 0.0f);
      const float lo2 = nd.corner[2] + ((c & 4) ? h : 0.0f);
      cnt[kRepLinksInOctant] += ch.cell_size > 0.0f && ch.cell_size <= h &&
                                ch.corner[0] >= lo0 && ch.corner[1] >= lo1 &&
                                ch.corner[2] >= lo2 && ch.corner[0] + ch.cell_size <= lo0 + h &&
                                ch.corner[1] + ch.cell_size <= lo1 + h &&
                                ch.corner[2] + ch.cell_size <= lo2 + h;
    }
  }
#pragma unroll
  for (int f = 0; f < kRepFields; ++f)
    if (f != kRepChainPastEnd) add_report(rep, f, cnt[f]);
}

// ---- compact form
struct CompactNode {
  uint32_t prefix;
  uint8_t level;  // level | depth << 4; 0xff: never written
  uint8_t node_mask;
  uint8_t child_set;
  uint8_t leaf_mask;
  uint32_t first_child;
};
static_assert(sizeof(CompactNode) == 12, "compact node layout");

// depth_of, for the cell sizes of an octree by way of their exponents: a
// quotient by 2^k lowers the exponent by k and keeps the fraction as long as
// it stays a normal number.
__device__ __forceinline__ int32_t depth_fast(float cell, float rg) {
  const uint32_t c = __float_as_uint(cell), r = __float_as_uint(rg);
  const int32_t k = static_cast<int32_t>(r >> 23) - static_cast<int32_t>(c >> 23);
  const bool normal = (c >> 23) - 1u < 254u && (r >> 23) - 1u < 254u;  // positive, finite
  if (normal && ((c ^ r) & 0x7fffffu) == 0 && k >= 0 && k <= 11) return k;
  return depth_of(cell, rg);
}

// axis_value, where one value in sight decodes to c: that value lies within
// one of (c - min) / range * 1024, so it is the one axis_value finds first.
__device__ __forceinline__ int32_t axis_fast(float c, int axis, int32_t level, float mn, float rg,
                                             float inv) {
  const auto decoded = [&](int32_t q) {  // decode_axis of the value itself
    return static_cast<float>(q) / 1024.0f * rg + mn;
  };
  const float est = (c - mn) * inv;
  if (est > -1.0f && est < 1024.0f) {
    const int32_t q = static_cast<int32_t>(rintf(est));
    const uint32_t grid = (1u << (level_shift(level) / 3u)) - 1u;
    if (q >= 0 && q <= 1023 && (static_cast<uint32_t>(q) & grid) == 0 &&
        __float_as_uint(decoded(q)) == __float_as_uint(c) && decoded(q - 1) != c &&
        decoded(q + 1) != c)
      return q;
  }
  return axis_value(c, axis, level, mn, rg);
}

// The header of a slot without its first-child index, or false when the
// slot has no exact compact form. w: the node's 15 words.
__device__ __forceinline__ bool compact_header(const int32_t (&w)[15], float mn, float rg,
                                               int32_t rl, CompactNode* cn) {
  *cn = CompactNode{};
  uint32_t set = 0, any = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) set |= (w[q] != 0 ? 1u : 0u) << q;
#pragma unroll
  for (int q = 0; q < 15; ++q) any |= static_cast<uint32_t>(w[q]);
  cn->child_set = static_cast<uint8_t>(set);
  if (any == 0) {
    cn->level = 0xff;
    return true;
  }
  const int32_t depth = depth_fast(__int_as_float(w[12]), rg);
  if (depth < 0 || rl + depth > 14) return false;
  const float inv = 1024.0f / rg;
  uint32_t pre = 0;
  bool on_grid = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int32_t q = axis_fast(__int_as_float(w[8 + a]), a, rl + depth, mn, rg, inv);
    on_grid &= q >= 0;
    pre |= split_by_3(static_cast<uint32_t>(q)) << a;
  }
  if (!on_grid || w[11] != __float_as_int(1.0f) || static_cast<uint32_t>(w[13]) > 255u ||
      static_cast<uint32_t>(w[14]) > 255u)
    return false;
  cn->prefix = pre;
  cn->level = static_cast<uint8_t>((rl + depth) | (depth << 4));
  cn->node_mask = static_cast<uint8_t>(w[13]);
  cn->leaf_mask = static_cast<uint8_t>(w[14]);
  return true;
}

// A segment's box and root level, as the kernels below need them for a slot.
struct SegInfo {
  float mn, rg;
  int32_t root_level;
};
struct SegTables {
  const int32_t* oct_start;
  int32_t n_seg;
  Boxes bx;
  const int32_t* seg_start;  // or nullptr: one segment
  const int32_t* n_unique;
  const uint8_t* prefix_n;
  __device__ __forceinline__ SegInfo of(int32_t seg) const {
    const int32_t sb = seg_start ? seg_start[seg] : 0;
    return {bx.min_of(seg), bx.range_of(seg), n_unique[seg] >= 2 ? prefix_n[sb] / 3 : 0};
  }
};

constexpr int kFmtTile = 512;  // slots per workgroup of the compact and expand kernels
constexpr int kFmtPer = kFmtTile / kFmtThreads;

// The headers of a thread's neighbouring slots, whose 120 bytes it loads for
// itself: a wave's are consecutive, and the caches pass every line on once.
struct TileSlots {
  CompactNode cn[kFmtPer];
  int32_t child[kFmtPer][8];
  uint32_t children = 0, bad = 0;
  __device__ __forceinline__ void form(const OctNode* __restrict__ nodes, int64_t g0, int32_t cnt,
                                       const SegTables& st) {
    const int32_t l0 = static_cast<int32_t>(threadIdx.x) * kFmtPer;
    int32_t w[kFmtPer][15];
    if (l0 + kFmtPer <= cnt) {
      __builtin_memcpy(w, nodes + g0 + l0, sizeof(w));
    } else {
#pragma unroll
      for (int u = 0; u < kFmtPer; ++u)
        if (l0 + u < cnt) __builtin_memcpy(w[u], nodes + g0 + l0 + u, sizeof(w[u]));
    }
    // (one segment holds the whole tile, as a rule)
    const int32_t seg0 = seg_of_slot(g0, st.oct_start, st.n_seg);
    const bool one = st.oct_start[seg0 + 1] >= g0 + cnt;
    SegInfo info = st.of(seg0);
#pragma unroll
    for (int u = 0; u < kFmtPer; ++u) {
      const int32_t l = l0 + u;
      cn[u] = CompactNode{};
      if (l >= cnt) continue;
      if (!one) info = st.of(seg_of_slot(g0 + l, st.oct_start, st.n_seg));
      bad += !compact_header(w[u], info.mn, info.rg, info.root_level, &cn[u]);
#pragma unroll
      for (int c = 0; c < 8; ++c) child[u][c] = w[u][c];
      children += __popc(cn[u].child_set);
    }
  }
};

// A tile's headers and children through LDS, to leave in whole lines. excl, before: the children before the tile and, in it,
// before the thread's slots. Children past child_cap are not stored.
constexpr int kFmtWords = kFmtTile * 11;  // eight children and a header of three words a slot
__device__ __forceinline__ void store_tile(TileSlots& slots, uint32_t* s_child, int64_t g0,
                                           int32_t cnt, uint32_t excl, uint32_t before,
                                           uint32_t total, uint32_t* __restrict__ out,
                                           int32_t* __restrict__ children, int64_t child_cap) {
  const int tid = threadIdx.x;
  uint32_t* s_head = s_child + kFmtTile * 8;
  uint32_t o = before;
#pragma unroll
  for (int u = 0; u < kFmtPer; ++u) {
    const int32_t l = tid * kFmtPer + u;
    if (l >= cnt) continue;
    slots.cn[u].first_child = excl + o;
    uint32_t hw[3];
    __builtin_memcpy(hw, &slots.cn[u], 12);
#pragma unroll
    for (int c = 0; c < 3; ++c) s_head[l * 3 + c] = hw[c];
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (slots.child[u][c] != 0) s_child[o++] = static_cast<uint32_t>(slots.child[u][c]);
  }
  __syncthreads();
  uint32_t* head = out + g0 * 3;
  for (int32_t q = tid; q < cnt * 3; q += kFmtThreads) head[q] = s_head[q];
  for (uint32_t q = tid; q < total; q += kFmtThreads)
    if (static_cast<int64_t>(excl) + q < child_cap)
      children[static_cast<int64_t>(excl) + q] = static_cast<int32_t>(s_child[q]);
}

// The compact form in one pass over the nodes: a tile's place in the child array
// comes from the two-level lookback. out and children may be null (the sizes
// only); children past child_cap are not stored. mail (host memory): [0] the
// children's total, [1] a wait gave up, [2] slots without an exact form exist
// (*bad counts them).
// What bounds it: 60 bytes a slot read and ~28 written; 0.99M slots take
// 25 us (27 with the nodes staged through LDS), where two passes over the nodes
// and three scan launches took 54, and the call 43 us instead of 208.
__global__ __launch_bounds__(kFmtThreads) void compact_kernel(
    const OctNode* __restrict__ nodes, int64_t k_total, SegTables st, uint64_t* __restrict__ flags,
    uint32_t* __restrict__ ctrl, uint32_t* __restrict__ out, int32_t* __restrict__ children,
    int64_t child_cap, unsigned long long* __restrict__ bad, uint32_t* __restrict__ mail) {
  __shared__ uint32_t s_words[kFmtWords];
  __shared__ uint32_t s_tmp[kFmtThreads / 64];
  __shared__ uint32_t s_excl;
  const uint32_t tag = ctrl[kCtrlEpoch] * 8u + kStageScan;
  if (stopped(ctrl, tag)) return;
  const int32_t t = blockIdx.x;  // in-order dispatch: see lookback_n
  const int64_t g0 = int64_t(t) * kFmtTile;
  const int32_t cnt = static_cast<int32_t>(min(int64_t(kFmtTile), k_total - g0));
  TileSlots slots;
  slots.form(nodes, g0, cnt, st);
  uint32_t total;
  const uint32_t before = block_excl_scan<kFmtThreads>(slots.children, s_tmp, &total);
  if (wave_id() == 0) {
    if (lane_id() == 0) flag_store(&flags[t], flag_pack(tag, kFlagAgg, total));
    bool late = false;
    const uint32_t prev = wave_lookback_groups(flags, flags + gridDim.x, t, 0, total, tag,
                                               wait_limit(ctrl), &late);
    if (lane_id() == 0) {
      if (late) {
        raise_timeout(ctrl, tag);
        mail[1] = 1u;
      }
      s_excl = prev;
      if (g0 + cnt == k_total) mail[0] = prev + total;
    }
  }
  if (slots.bad) {
    atomicAdd(bad, static_cast<unsigned long long>(slots.bad));
    mail[2] = 1u;
  }
  __syncthreads();
  if (!out || !children) return;
  store_tile(slots, s_words, g0, cnt, s_excl, before, total, out, children, child_cap);
}

// The compact form in two passes over the nodes, whose tiles wait for nothing. For
// a pipeline's slots, as launches with waits of two frames may not overlap, and
// this one is outside their order; and for calls that may yet be refused, as the
// second pass knows all counts before it stores. Tiles form at most kCompactGroups groups of
// neighbours, a workgroup each in the first pass: tile_children[t], and per group
// {children, slots without an exact form}. The second pass sums the groups before
// its own and its group's tiles before its own.
// What bounds them: 60 bytes a slot read twice and ~28 written; 0.99M slots take
// 15 and 22 us, the call 53 where the one pass takes 43.
constexpr int32_t kCompactGroups = 2048;
__host__ __device__ __forceinline__ int32_t tiles_per_group(int32_t tiles) {
  return (tiles + kCompactGroups - 1) / kCompactGroups;
}
__global__ __launch_bounds__(kFmtThreads) void compact_count_kernel(
    const OctNode* __restrict__ nodes, int64_t k_total, SegTables st, int32_t tiles,
    uint2* __restrict__ groups, uint32_t* __restrict__ tile_children) {
  __shared__ uint32_t s_tmp[2 * (kFmtThreads / 64)];
  const int32_t per = tiles_per_group(tiles);
  const int32_t t0 = static_cast<int32_t>(blockIdx.x) * per;
  uint2 sum = make_uint2(0u, 0u);
  for (int32_t t = t0; t < min(t0 + per, tiles); ++t) {
    const int64_t g0 = int64_t(t) * kFmtTile;
    const int32_t cnt = static_cast<int32_t>(min(int64_t(kFmtTile), k_total - g0));
    TileSlots slots;
    slots.form(nodes, g0, cnt, st);
    const uint32_t c = wave_sum(slots.children), b = wave_sum(slots.bad);
    if (lane_id() == 0) {
      s_tmp[2 * wave_id()] = c;
      s_tmp[2 * wave_id() + 1] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t n = 0;
#pragma unroll
      for (int w = 0; w < kFmtThreads / 64; ++w) {
        n += s_tmp[2 * w];
        sum.y += s_tmp[2 * w + 1];
      }
      tile_children[t] = n;
      sum.x += n;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) groups[blockIdx.x] = sum;
}

// mail (host memory): [0] the children's total, [2] the number of slots without
// an exact form. A grid of one with out null: these alone. Where there are such
// slots, or more children than child_cap, nothing is stored.
__global__ __launch_bounds__(kFmtThreads) void compact_write_kernel(
    const OctNode* __restrict__ nodes, int64_t k_total, SegTables st, int32_t tiles,
    const uint2* __restrict__ groups, const uint32_t* __restrict__ tile_children,
    uint32_t* __restrict__ out, int32_t* __restrict__ children, int64_t child_cap,
    uint32_t* __restrict__ mail) {
  __shared__ uint32_t s_words[kFmtWords];
  __shared__ uint32_t s_tmp[kFmtThreads / 64];
  __shared__ uint32_t s_sum[3];  // children before the tile, all children, bad slots
  const int tid = threadIdx.x;
  const int32_t t = blockIdx.x;
  const int64_t g0 = int64_t(t) * kFmtTile;
  const int32_t cnt = static_cast<int32_t>(min(int64_t(kFmtTile), k_total - g0));
  if (tid < 3) s_sum[tid] = 0;
  const int32_t per = tiles_per_group(tiles);
  const int32_t own = t / per, n_groups = (tiles + per - 1) / per;
  uint32_t before = 0, all = 0, bad = 0;
  for (int32_t q = tid; q < n_groups; q += kFmtThreads) {
    const uint2 g = groups[q];
    all += g.x;
    bad += g.y;
    if (q < own) before += g.x;
  }
  for (int32_t q = own * per + tid; q < t; q += kFmtThreads) before += tile_children[q];
  TileSlots slots;
  if (out) slots.form(nodes, g0, cnt, st);
  __syncthreads();
  before = wave_sum(before);
  all = wave_sum(all);
  bad = wave_sum(bad);
  if (lane_id() == 0) {
    atomicAdd(&s_sum[0], before);
    atomicAdd(&s_sum[1], all);
    atomicAdd(&s_sum[2], bad);
  }
  __syncthreads();
  if (t == 0 && tid == 0) {
    mail[0] = s_sum[1];
    mail[2] = s_sum[2];
  }
  if (!out || s_sum[2] != 0 || static_cast<int64_t>(s_sum[1]) > child_cap) return;
  uint32_t total;
  const uint32_t first = block_excl_scan<kFmtThreads>(slots.children, s_tmp, &total);
  store_tile(slots, s_words, g0, cnt, s_sum[0], first, total, out, children, child_cap);
}

// 60-byte nodes from the compact form, a tile's through LDS so that whole
// lines leave. Child indices at or past n_children read as 0.
// What bounds it: 60 bytes a slot written and ~28 read; 0.99M slots take 16 us
// (26 with the 60 bytes stored by each thread for itself).
__global__ __launch_bounds__(kFmtThreads) void expand_kernel(
    const CompactNode* __restrict__ in, const int32_t* __restrict__ children, int64_t n_children,
    const int32_t* __restrict__ oct_start, int32_t n_seg, Boxes bx, OctNode* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) int32_t s_words[kFmtTile * 15];
  const int tid = threadIdx.x;
  const int64_t k_total = oct_start[n_seg];
  for (int64_t g0 = int64_t(blockIdx.x) * kFmtTile; g0 < k_total;
       g0 += int64_t(gridDim.x) * kFmtTile) {
    const int32_t cnt = static_cast<int32_t>(min(int64_t(kFmtTile), k_total - g0));
    const int32_t seg0 = seg_of_slot(g0, oct_start, n_seg);
    const bool one = oct_start[seg0 + 1] >= g0 + cnt;
#pragma unroll
    for (int u = 0; u < kFmtTile / kFmtThreads; ++u) {
      const int32_t l = u * kFmtThreads + tid;
      if (l >= cnt) continue;
      const CompactNode cn = in[g0 + l];
      int32_t* w = s_words + l * 15;
      int64_t o = cn.first_child;
      int32_t ch[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        ch[q] = 0;
        if (!((cn.child_set >> q) & 1u)) continue;
        // a malformed node (offset outside [0, n_children)) reads no memory
        if (o < n_children) ch[q] = children[o];
        ++o;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = ch[q];
      const bool written = cn.level != 0xff;
      const int32_t seg = one ? seg0 : seg_of_slot(g0 + l, oct_start, n_seg);
      const float mn = bx.min_of(seg), rg = bx.range_of(seg);
      const uint32_t sh = static_cast<uint32_t>(cn.level >> 4) & 31u;
      w[8] = written ? __float_as_int(decode_axis(cn.prefix, 0, mn, rg)) : 0;
      w[9] = written ? __float_as_int(decode_axis(cn.prefix, 1, mn, rg)) : 0;
      w[10] = written ? __float_as_int(decode_axis(cn.prefix, 2, mn, rg)) : 0;
      w[11] = written ? __float_as_int(1.0f) : 0;
      w[12] = written ? __float_as_int(rg / static_cast<float>(static_cast<int32_t>(1u << sh))) : 0;
      w[13] = written ? cn.node_mask : 0;
      w[14] = written ? cn.leaf_mask : 0;
    }
    __syncthreads();
    int32_t* dst = reinterpret_cast<int32_t*>(out + g0);
    const int32_t words = cnt * 15;
    for (int32_t q = tid * 4; q < words; q += kFmtThreads * 4) {
      if (q + 4 <= words) {
        const int4 v = *reinterpret_cast<const int4*>(s_words + q);
        __builtin_memcpy(dst + q, &v, 16);
      } else {
        for (int32_t c = q; c < words; ++c) dst[c] = s_words[c];
      }
    }
    __syncthreads();
  }
}

}  // namespace

void launch_seg_roots(const uint32_t* codes, const uint8_t* prefix_n, const int32_t* n_unique,
                      const int32_t* seg_start, int32_t n_seg, int32_t* root_level,
                      uint32_t* root_code, hipStream_t s) {
  if (n_seg <= 0) return;
  seg_roots_kernel<<<(n_seg + 255) / 256, 256, 0, s>>>(codes, prefix_n, n_unique, seg_start,
                                                       n_seg, root_level, root_code);
}

void launch_validate(const OctNode* nodes, const int32_t* edge, const int32_t* offs,
                     const int32_t* n_unique, const int32_t* oct_start, const int32_t* seg_start,
                     int32_t n_seg, const float* smin, const float* srg, float mn1, float rg1,
                     const int32_t* root_level, const uint32_t* root_code, uint8_t* cov,
                     unsigned long long* rep, hipStream_t s) {
  if (n_seg <= 0) return;
  dim3 grid(64, std::min(n_seg, 1024));
  cover_kernel<<<grid, kFmtThreads, 0, s>>>(edge, offs, n_unique, oct_start, seg_start, n_seg,
                                            cov, rep);
  const Boxes bx{smin, srg, mn1, rg1};
  validate_kernel<<<kFmtGrid, kFmtThreads, 0, s>>>(nodes, cov, oct_start, n_seg, bx, root_level,
                                                   root_code, rep);
}

int64_t compact_tiles(int64_t k_total) { return (k_total + kFmtTile - 1) / kFmtTile; }

static SegTables seg_tables(const CompactSource& c) {
  return {c.oct_start, c.n_seg, Boxes{c.smin, c.srg, c.mn1, c.rg1}, c.seg_start, c.n_unique,
          c.prefix_n};
}

void launch_compact(const CompactSource& c, uint64_t* flags, uint32_t* ctrl, void* out,
                    int32_t* children, int64_t child_cap, unsigned long long* bad, uint32_t* mail,
                    hipStream_t s) {
  if (c.n_seg <= 0 || c.k_total <= 0) return;
  compact_kernel<<<static_cast<uint32_t>(compact_tiles(c.k_total)), kFmtThreads, 0, s>>>(
      c.nodes, c.k_total, seg_tables(c), flags, ctrl, static_cast<uint32_t*>(out), children,
      child_cap, bad, mail);
}

int64_t compact_words(int64_t k_total) { return 2 * kCompactGroups + compact_tiles(k_total); }

void launch_compact_no_wait(const CompactSource& c, uint32_t* words, void* out, int32_t* children,
                            int64_t child_cap, uint32_t* mail, hipStream_t s) {
  if (c.n_seg <= 0 || c.k_total <= 0) return;
  const SegTables st = seg_tables(c);
  const int32_t tiles = static_cast<int32_t>(compact_tiles(c.k_total));
  const int32_t per = tiles_per_group(tiles);
  uint2* groups = reinterpret_cast<uint2*>(words);
  uint32_t* tile_children = words + 2 * kCompactGroups;
  compact_count_kernel<<<(tiles + per - 1) / per, kFmtThreads, 0, s>>>(c.nodes, c.k_total, st,
                                                                      tiles, groups, tile_children);
  compact_write_kernel<<<out ? tiles : 1, kFmtThreads, 0, s>>>(
      c.nodes, c.k_total, st, tiles, groups, tile_children, static_cast<uint32_t*>(out), children,
      child_cap, mail);
}

void launch_expand(const void* in, const int32_t* children, int64_t n_children,
                   const int32_t* oct_start, int32_t n_seg, const float* smin, const float* srg,
                   float mn1, float rg1, OctNode* out, hipStream_t s) {
  if (n_seg <= 0) return;
  const Boxes bx{smin, srg, mn1, rg1};
  expand_kernel<<<kFmtGrid, kFmtThreads, 0, s>>>(static_cast<const CompactNode*>(in), children,
                                                 n_children, oct_start, n_seg, bx, out);
}

}  // namespace ocp
