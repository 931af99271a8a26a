// Stage 7: octree nodes from the radix tree -
// ProcessOctNode and ProcessLinkLeaf of include/shared/oct.h:24-134, driven
// by kernels/07_octree.cpp:5-57 - with the sequential (ascending index)
// semantics of the reference CPU path, in one pass.
//
// The reference's chains overlap: the offsets P are an inclusive scan
// (kernels/06_partial_sum.cpp) but P[i] is used as the first slot of chain
// i, so run sequentially the last writer of a field wins. The kernel gives
// every node slot exactly one writer that computes its final 60 bytes:
//
//  * Chain i (e[i] > 0) covers slots P[i] .. P[i]+e[i]-1. Non-empty chains
//    start strictly later as i grows, so chain i always owns its first slot
//    and owns slot P[i]+j unless a later chain covers it. The owner writes
//    the corner and cell size of step j (oct.h:44-57, 76-88).
//  * Make-phase child links into slot s come from the chains covering s:
//    chain q writes children[c] = s-1 there (oct.h:41-51), so those links
//    need no ordering, only the union of their child indices. The first
//    slot P[a] of chain a additionally receives the top links of the
//    non-empty chains whose parent walk (oct.h:61-73) ends at a, and the
//    leaf links (oct.h:92-134) of every node whose walk ends at a. Those
//    nodes are a's group: a and the e == 0 internal nodes below it, at most
//    two levels deep because prefix lengths grow strictly down the tree and
//    one octree level spans three of them. Per child index the write that
//    comes last in the sequential order stays: make writes by (chain, step),
//    every link write after every make write, links by (node, side).
//  * The root group follows parent[] rather than node 0's own children:
//    node 0 is the reference's short-range root (04_radix_tree.cpp:63-65),
//    and the nodes whose parent is 0 are the children of the true root.
//  * Slots no chain covers stay zero; they are written like any other, so
//    the node buffer needs no zero fill.
//  * child_leaf_mask only ever sees AND-NOT on a zeroed word (oct.h:20), so
//    it is 0; child_node_mask is the OR of the make-phase link bits.
//
// Layout of the work: every node slot belongs to one tile of 512 BRT nodes,
// the one that holds the node at which the inclusive scan reaches the slot
// (the slots P[i0-1]+1 .. P[i0+511]; slot 0 to the first tile, the slots past
// the last node's P to the last). A tile's chains start in its own slots.
//  1. One thread per node pushes what the node writes into LDS columns, one
//     per slot: its leaf links into the slot its walk up parent[] ends at
//     (itself for a chain), a chain's top link into the slot the walk from
//     its parent ends at, a chain's step links and its geometry into the
//     slots it covers. An entry is 64 bits, order key above value, kept by an
//     LDS atomic max, so the last writer of the sequential order stays. Nodes
//     before the tile whose chains reach into its slots are pushed by one
//     wave that scans back over them.
//  2. A walk that leaves the tile pushes nothing. Instead, a node of the tile
//     whose walk ends in it lists its internal children outside the tile, and
//     one thread per listed child walks that part of the group downwards in
//     global memory. Such a node spans a tile end, and the nodes spanning one
//     are nested with different prefix lengths, so at most 124 are listed.
//  3. One thread per slot assembles the node, packs it over the columns, and the
//     tile's nodes leave as consecutive 16-byte stores.
// A tile with more slots than columns takes them in several rounds.
//
// The per-stage entries (k_MakeOctNodes, k_LinkLeafNodes: include/cuda/kernels/
// 07_octree.cuh:7-28) are the same kernel doing one half of the pushes into
// nodes that it reads and writes whole, where a kernel before it has found the
// caller's arrays to be what a build's are (check_kernel); for any others, as
// offsets that are not the inclusive scan, or codes that repeat or have more than
// 30 bits, it scatters order keys by global atomics and a kernel after it resolves
// them. Make has no children arrays: see check_kernel. For 2M points make takes 16
// us of check, 30 of the tiled kernel and 5 of the idle resolve, link 13, 30 and 5;
// for arrays of another form they take 131 and 197 us (117 and 182 when the scatter
// and the resolve, without a check, served every array).
//
// What bounds it: how many tiles share a CU while each waits for its loads, its
// barriers and the walks of its listed children (a chain of up to four dependent
// loads that one wave makes while the others wait). 10M uniform points take
// 135 us, 2^24 clustered ones 57; 24 bytes a node read and 60 a slot written are
// 104 us of the former at the rate of a large copy. Before the nodes of builds
// that size were stored past the caches (oct_stream), 152 us and 59. 312 columns of 64 bytes are
// what lets six tiles share a CU's LDS, as 60 registers do; with 80 bytes a
// column (an own word for the mask) and nodes finished where their column lay,
// five did, in 174 us and 67. Four tiles by registers took 188; 256 columns, with
// which more tiles need a second round, 155 and 68. One wave walking the listed
// children while three push was slower (182), and so were 256 nodes a tile, one
// per thread, and stores of 60 bytes a lane (244), two per thread in 512-thread
// workgroups (212), and a lane per chain that walked its group down, read its
// neighbours' chains and resolved keys into values (250).
//
// Edge counts are at most 10 (prefix lengths are at most 31 for 30-bit
// codes), so a chain spans at most 10 slots.
#include "ocp_internal.hpp"

namespace ocp {
namespace {

constexpr int32_t kMaxEdge = 10;
constexpr uint32_t kMaxPrefix = 31;                // of 30-bit codes (a node of one code)
constexpr uint32_t kCodeEnd = 1u << kMortonBits;  // what an owner word and third() hold
constexpr int kThreads = 256;
constexpr int kCols = 312;      // slots per round; a tile of 512 nodes has ~240
constexpr int kCodeHalo = 32;   // codes staged on either side of a tile
constexpr int kMaxOutside = 128;
// A node's step of a walk up, 16 bits: kHead + slot of the tile where the walk
// ends (a chain's first slot, node 0's slot 0), else the parent's place in the
// tile, kOutside if it has none.
constexpr uint32_t kHead = 0x8000u;
constexpr uint32_t kOutside = 0x4000u;
constexpr uint32_t kNoSlot = 0xffffffffu;

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef int32_t v4i_any __attribute__((ext_vector_type(4), aligned(4)));

struct SegBind {
  OctNode* nodes;
  int32_t k;
  int32_t m;
  const uint32_t* codes;
  const uint8_t* pn;
  const uint8_t* hl;
  const uint8_t* hr;
  const int32_t* lc;
  const int32_t* par;
  const int32_t* e;
  const int32_t* p;
  float mn;
  float rg;
};

__device__ __forceinline__ uint32_t child_of(uint32_t code, int32_t level) {
  return (code >> (static_cast<uint32_t>(kMortonBits - 3 * level) & 31u)) & 7u;
}
// Order of the sequential program: make writes by (chain, step), every link
// write after every make write, links by (node, side).
__device__ __forceinline__ uint32_t make_key(int32_t chain, int32_t step) {
  return static_cast<uint32_t>((chain << 4) | step) + 1u;
}
__device__ __forceinline__ uint32_t link_key(int32_t node, int side) {
  return 0x80000000u | static_cast<uint32_t>((node << 1) | side);
}

typedef unsigned long long u64;

// The columns of the slots [base, base + n), n <= kCols: eight 8-byte words a
// slot, the last writer of each child index (order key << 32 | value, 0: none),
// turned by one every four slots so that one child index of many slots spreads
// over the LDS banks. The finished nodes take the columns' place.
constexpr int kColWords = 8;
__device__ __forceinline__ uint32_t col_word(uint32_t r, uint32_t which) {
  return r * kColWords + ((which + (r >> 2)) & 7u);
}
struct Columns {
  lds_ptr<u64> child;
  lds_ptr<u64> owner;     // chain + 1 << 34 | level << 30 | code, 0: no chain
  lds_ptr<uint32_t> mask;  // child-node masks, a byte each
  int32_t base;
  int32_t n;
  __device__ __forceinline__ void put(uint32_t slot, uint32_t which, uint32_t key,
                                      int32_t value) const {
    const uint32_t r = slot - static_cast<uint32_t>(base);
    if (r < static_cast<uint32_t>(n))
      __hip_atomic_fetch_max(child + col_word(r, which),
                             (static_cast<u64>(key) << 32) | static_cast<uint32_t>(value),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // A make-phase write also sets its bit of the mask.
  __device__ __forceinline__ void put_make(uint32_t slot, uint32_t which, uint32_t key,
                                           int32_t value) const {
    const uint32_t r = slot - static_cast<uint32_t>(base);
    if (r >= static_cast<uint32_t>(n)) return;
    put(slot, which, key, value);
    __hip_atomic_fetch_or(mask + (r >> 2), 1u << ((r & 3u) * 8u + which),
                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // Chain i: the slots p .. p + e - 1 with their geometry, and its step links
  // (oct.h:41-51) into all but the first.
  __device__ __forceinline__ void cover(int32_t i, int32_t p, int32_t e, uint32_t code,
                                        int32_t level) const {
    const int32_t steps = min(e, kMaxEdge);
    for (int32_t j = 0; j < steps; ++j) {
      const uint32_t r = static_cast<uint32_t>(p + j - base);
      if (r >= static_cast<uint32_t>(n)) continue;
      __hip_atomic_fetch_max(owner + r,
                             (static_cast<u64>(i + 1) << 34) |
                                 (static_cast<u64>(level - j) << 30) | code,
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (j > 0)
        put_make(static_cast<uint32_t>(p + j), child_of(code, level - (j - 1)),
                 make_key(i, j - 1), p + j - 1);
    }
  }
};

// The part of slot `slot`'s group from node x down, read from global memory:
// top links of chains, leaf links and children of e == 0 nodes. A step takes
// an e == 0 node's two children, which are neighbours in every array (a leaf
// is a code, an internal child a node, of index left_child + side), with all
// of their loads in flight together, so the chain of dependent loads is one
// per e == 0 node. Such nodes are at most three levels deep: prefix lengths
// grow strictly down the tree and one octree level spans three of them, so
// three pending ones suffice and seven steps are the most. The link phase, on a
// caller's arrays, has a bound all the same (in the build's own, of unique codes,
// it would cost 0.5 us of 133).
constexpr int kMaxSteps = 16;
struct SubNode {
  int32_t x, lc;
  uint32_t flags;  // level | has_leaf_left << 8 | has_leaf_right << 9
};
template <bool MAKE>
__device__ __forceinline__ void push_subgroup(const SegBind& b, const Columns& cols, int32_t x,
                                              uint32_t slot) {
  SubNode cur, s0{}, s1{}, s2{};  // s0..s2: pending, s0 on top
  int pending = 0;
  {
    const int32_t e = b.e[x];
    const int32_t p = b.p[x];
    const uint32_t code = b.codes[x];
    const int32_t level = third(b.pn[x]);
    cur = {x, b.lc[x],
           static_cast<uint32_t>(level) | (b.hl[x] ? 256u : 0u) | (b.hr[x] ? 512u : 0u)};
    if (MAKE && e > 0)
      cols.put_make(slot, child_of(code, level - e + 1), make_key(x, e - 1), p + e - 1);
    if (e != 0) return;
  }
  for (int step = 0; MAKE || step < kMaxSteps; ++step) {
    int32_t e[2], p[2], lc[2];
    uint32_t code[2];
    uint8_t pn[2], hl[2], hr[2];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int32_t node = min(cur.lc + side, b.m - 1);  // (a leaf may be key m)
      code[side] = b.codes[cur.lc + side];
      e[side] = b.e[node];
      p[side] = b.p[node];
      lc[side] = b.lc[node];
      pn[side] = b.pn[node];
      hl[side] = b.hl[node];
      hr[side] = b.hr[node];
    }
    const int32_t level = static_cast<int32_t>(cur.flags & 15u);
    const SubNode at = cur;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int32_t ch = at.lc + side;
      const int32_t lv = third(pn[side]);
      if (at.flags & (256u << side)) {
        cols.put(slot, child_of(code[side], level + 1), link_key(at.x, side), ch);
      } else if (e[side] > 0) {
        if (MAKE) cols.put_make(slot, child_of(code[side], lv - e[side] + 1), make_key(ch, e[side] - 1),
                      p[side] + e[side] - 1);
      } else if (e[side] == 0 && pending < 3) {
        s2 = s1;
        s1 = s0;
        s0 = {ch, lc[side],
              static_cast<uint32_t>(lv) | (hl[side] ? 256u : 0u) | (hr[side] ? 512u : 0u)};
        ++pending;
      }
    }
    if (pending == 0) break;
    cur = s0;
    s0 = s1;
    s1 = s2;
    --pending;
  }
}

// The writes of node i as order keys in the child words of the nodes, kept by an
// atomic max: the per-stage entries' path for arrays of any form, finished by
// resolve_kernel.
__device__ __forceinline__ void put_word(const OctArgs& a, int32_t slot, uint32_t which,
                                         uint32_t key) {
  if (slot >= 0 && slot < a.k_host)
    atomicMax(reinterpret_cast<uint32_t*>(&a.nodes[slot].children[which]), key);
}
__device__ __forceinline__ void put_make_word(const OctArgs& a, int32_t slot, uint32_t which,
                                              uint32_t key) {
  if (slot < 0 || slot >= a.k_host) return;
  put_word(a, slot, which, key);
  atomicOr(&a.nodes[slot].child_node_mask, 1 << which);
}
// The node that the walk of oct.h:61-73 from node i's parent ends at (at most
// 31 hops; node 0 is its own parent). A hop's two loads are in flight together.
__device__ __forceinline__ int32_t make_head(const OctArgs& a, int32_t i) {
  int32_t h = a.parent[i];
  for (int hop = 0; hop < 31; ++hop) {
    const int32_t e = a.edge[h], up = a.parent[h];
    if (e != 0 || up == h) break;
    h = up;
  }
  return h;
}
template <bool MAKE>
__device__ __forceinline__ void scatter_node(const OctArgs& a, int32_t i) {
  if (i >= a.n_brt_host) return;
  if constexpr (MAKE) {
    const int32_t e = a.edge[i];
    if (i == 0 || e <= 0) return;
    const int32_t p = a.offsets[i];
    const int32_t level = a.prefix_n[i] / 3;
    const uint32_t code = a.codes[i];
    for (int32_t j = 0; j < e - 1; ++j)
      put_make_word(a, p + j + 1, child_of(code, level - j), make_key(i, j));
    put_make_word(a, a.offsets[make_head(a, i)], child_of(code, level - e + 1),
                  make_key(i, e - 1));
  } else {
    int32_t head = -1;
    for (int side = 0; side < 2; ++side) {
      if (!(side == 0 ? a.has_leaf_left[i] : a.has_leaf_right[i])) continue;
      if (head < 0) {
        // oct.h:111-113, stopped at node 0 and after 64 hops
        head = i;
        for (int hop = 0; hop < 64 && a.edge[head] == 0 && head != 0; ++hop)
          head = a.parent[head];
      }
      const int32_t slot = a.offsets[head];
      const uint32_t which =
          child_of(a.codes[a.left_child[i] + side], a.prefix_n[i] / 3 + 1);
      put_word(a, slot, which, link_key(i, side));
      if (slot >= 0 && slot < a.k_host)
        atomicAnd(&a.nodes[slot].child_leaf_mask, ~(1 << which));
    }
  }
}

// What a launch does: the whole stage (storing its nodes past the caches or not:
// a template, for as a branch the two stores are merged into an ordinary one), or
// one of its two per-stage entries on nodes that the caller prepared.
enum OctPhase { kWhole, kWholeStreamed, kMakePhase, kLinkPhase };

template <bool SINGLE, OctPhase PHASE>
__global__ __launch_bounds__(kThreads) void oct_build_kernel(
    OctArgs a, SegView sv, const int32_t* __restrict__ tile_start, OctSingle one) {
  constexpr int T = kOctTile;
  constexpr int NPT = T / kThreads;
  constexpr bool MAKE = PHASE != kLinkPhase, LINK = PHASE != kMakePhase;
  constexpr bool WHOLE = PHASE == kWhole || PHASE == kWholeStreamed;
  __shared__ __attribute__((aligned(16))) u64 s_child[kColWords * kCols];
  __shared__ u64 s_owner[kCols];
  __shared__ uint32_t s_mask[kCols / 4];
  __shared__ uint16_t s_walk[T];
  __shared__ uint32_t s_code[T + 2 * kCodeHalo];
  __shared__ int32_t s_out[kMaxOutside];  // listed children ...
  __shared__ uint16_t s_out_slot[kMaxOutside];  // ... and their slots of the tile
  __shared__ uint32_t s_nout;

  const TileRef r = find_tile(tile_start, sv.n_seg, xcd_tile(blockIdx.x, gridDim.x));
  if constexpr (!WHOLE) {
    if (*a.form == a.form_id) {  // (arrays of another form than a build's)
      for (int u = 0; u < NPT; ++u)
        scatter_node<MAKE>(a, r.local * T + u * kThreads + static_cast<int32_t>(threadIdx.x));
      return;
    }
  }
  // The segment's scalars are loaded together before any is tested: one
  // round trip instead of one per value.
  // (The launcher guarantees these pointers; the build writes them all.)
  const int32_t m_seg = WHOLE ? a.n_unique[r.seg] - 1 : a.n_brt_host;
  const int32_t k_seg = WHOLE ? a.kalloc[r.seg] : a.k_host;
  const uint32_t fits = !WHOLE ? 1u
                        : SINGLE        ? (static_cast<uint32_t>(k_seg) <= one.k_cap ? 1u : 0u)
                                        : a.ctrl[kCtrlOctOk];
  const int32_t node_base = SINGLE || !WHOLE ? 0 : a.oct_start[r.seg];
  const int32_t sb = seg_begin(sv, r.seg);
  const float seg_mn = seg_min(sv, r.seg);
  const float seg_rg = seg_range(sv, r.seg);
  const int32_t i0 = r.local * T;
  // One test after all the loads (an early return per value would hold the
  // loads after it back): the nodes fit, the tile has nodes (a single-key
  // segment still has its root), the segment has slots and a valid base.
  // After a lookback time-out the inputs are not valid.
  const uint32_t stop = WHOLE ? a.ctrl[kCtrlTimeout] : 0u;
  if (SINGLE && i0 == 0 && threadIdx.x == 0) {
    // What the offsets kernel does for several segments (a launch of ~5 us).
    const uint32_t tiles = a.ctrl[kCtrlMsdTiles];
    const uint32_t slots = static_cast<uint32_t>(k_seg);
    one.oct_start[0] = 0;
    one.oct_start[1] = k_seg;
    one.ctrl[kCtrlOctTotal] = slots;
    one.ctrl[kCtrlOctOk] = fits;
    one.mail[kCtrlOctTotal] = slots;
    one.mail[kCtrlOctOk] = fits;
    one.mail[kCtrlTimeout] = stop;
    one.mail[kCtrlMsdTiles] = tiles;
    one.mail[kCtrlWords] = static_cast<uint32_t>(m_seg + 1);
    one.mail[kCtrlWords + kMailSegs] = slots;
  }
  if (fits == 0 || stop != 0 || (i0 >= m_seg && !(i0 == 0 && m_seg == 0)) || k_seg < 1 ||
      node_base < 0)
    return;
  SegBind b;
  b.m = m_seg;
  b.nodes = a.nodes + node_base;
  b.k = k_seg;
  b.codes = a.codes + sb;
  b.pn = a.prefix_n + sb;
  b.hl = a.has_leaf_left + sb;
  b.hr = a.has_leaf_right + sb;
  b.lc = a.left_child + sb;
  b.par = a.parent + sb;
  b.e = a.edge + sb;
  b.p = a.offsets + sb;
  b.mn = seg_mn;
  b.rg = seg_rg;

  // The slots of the tile.
  const int32_t i_end = min(i0 + T, b.m);
  int32_t p_before = i0 > 0 ? b.p[i0 - 1] : -1;
  int32_t s_end = i_end >= b.m ? b.k : b.p[i_end - 1] + 1;
  if constexpr (!WHOLE) {
    // The caller's slots bound every access, and those past the last chain
    // stay as they are.
    if (i_end >= b.m) s_end = b.p[b.m - 1] + kMaxEdge;
    p_before = max(p_before, -1);
    s_end = min(s_end, b.k);
  }
  const int32_t root_level = b.m >= 1 ? third(b.pn[0]) : 0;

  if (p_before + 1 >= s_end) return;  // a tile without slots

  Columns cols;
  cols.child = as_lds<u64>(s_child);
  cols.owner = as_lds<u64>(s_owner);
  cols.mask = as_lds<uint32_t>(s_mask);
  const int32_t slot_0 = p_before + 1;

  for (cols.base = slot_0; cols.base < s_end; cols.base += kCols) {
    cols.n = min(kCols, s_end - cols.base);
    // (opaque: the compiler would keep every address of a round for the next)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    // (loaded in every round, of which a tile rarely has a second, so that
    // they hold no register beyond the pushes)
    // This thread's nodes, and for the last wave one of the 64 nodes before the
    // tile: all loads in flight together.
    int32_t p[NPT], e[NPT], lc[NPT], par[NPT];
    uint32_t code[NPT];
    uint8_t pn[NPT], hl[NPT], hr[NPT];
    if (i0 + T <= b.m) {
#pragma unroll
      for (int u = 0; u < NPT; ++u) {
        const int32_t i = i0 + u * kThreads + tid;
        p[u] = b.p[i];
        e[u] = b.e[i];
        par[u] = b.par[i];
        code[u] = b.codes[i];
        pn[u] = b.pn[i];
        if constexpr (LINK) {
          lc[u] = b.lc[i];
          hl[u] = b.hl[i];
          hr[u] = b.hr[i];
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < NPT; ++u) {
        const int32_t i = i0 + u * kThreads + tid;
        p[u] = e[u] = lc[u] = 0;
        par[u] = 0x7fffffff;
        code[u] = 0;
        pn[u] = hl[u] = hr[u] = 0;
        if (i < b.m) {
          p[u] = b.p[i];
          e[u] = b.e[i];
          par[u] = b.par[i];
          pn[u] = b.pn[i];
          if constexpr (LINK) {
            lc[u] = b.lc[i];
            hl[u] = b.hl[i];
            hr[u] = b.hr[i];
          }
        }
        if (LINK ? i <= b.m : i < b.m) code[u] = b.codes[i];  // (make: as many codes as nodes)
      }
    }
    uint32_t code_halo = 0;
    if (LINK && tid < 2 * kCodeHalo) {
      const int32_t g = tid < kCodeHalo ? i0 - kCodeHalo + tid : i0 + T + tid - kCodeHalo;
      if (g >= 0 && g <= b.m) code_halo = b.codes[g];
    }
    int32_t back_e = 0, back_p = 0;
    const int32_t back_q = i0 - 1 - static_cast<int32_t>(lane_id());
    const bool back_wave = MAKE && wave_id() == kThreads / 64 - 1 && i0 > 0;
    if (back_wave && back_q >= 1) {
      back_e = b.e[back_q];
      back_p = b.p[back_q];
    }
    for (int q = tid; q < kColWords * kCols / 2; q += kThreads)
      reinterpret_cast<v4i*>(s_child)[q] = v4i{0, 0, 0, 0};
    for (int q = tid; q < kCols; q += kThreads) s_owner[q] = 0;
    static_assert(kCols % 4 == 0 && kCols / 4 <= kThreads, "masks");
    if (tid < kCols / 4) s_mask[tid] = 0;
#pragma unroll
    for (int u = 0; u < NPT; ++u) {
      const int32_t i = i0 + u * kThreads + tid;
      const bool head = i < b.m && (e[u] > 0 || i == 0);
      const uint32_t up = static_cast<uint32_t>(par[u] - i0);
      s_walk[u * kThreads + tid] = static_cast<uint16_t>(
          head ? kHead | (static_cast<uint32_t>(p[u] - slot_0) & 0x3fffu)
               : min(up, kOutside));
      s_code[kCodeHalo + u * kThreads + tid] = code[u];
    }
    if (tid < kCodeHalo) s_code[tid] = code_halo;
    else if (tid < 2 * kCodeHalo) s_code[T + tid] = code_halo;
    if (tid == 0) s_nout = 0;
    __syncthreads();

#pragma unroll
    for (int u = 0; u < NPT; ++u) {
      const int32_t i = i0 + u * kThreads + tid;
      if (i >= b.m) continue;
      const int32_t level = third(pn[u]);
      // The walk up from the node's parent: the slot it ends at, or kNoSlot
      // where it leaves the tile.
      uint32_t up = kNoSlot;
      if (i > 0) {
        uint32_t h = min(static_cast<uint32_t>(par[u] - i0), kOutside);
        for (int hop = 0; hop < 8 && h < static_cast<uint32_t>(T); ++hop) h = s_walk[h];
        if (h - kHead <= 0x3fffu) up = static_cast<uint32_t>(slot_0) + (h - kHead);
      }
      const uint32_t slot = (e[u] > 0 || i == 0) ? static_cast<uint32_t>(p[u]) : up;
      if (LINK && slot != kNoSlot) {
#pragma unroll
        for (int side = 0; side < 2; ++side) {
          const int32_t ch = lc[u] + side;
          if (side == 0 ? hl[u] != 0 : hr[u] != 0) {
            const uint32_t rel = static_cast<uint32_t>(ch - i0 + kCodeHalo);
            const uint32_t c =
                rel < static_cast<uint32_t>(T + 2 * kCodeHalo) ? s_code[rel] : b.codes[ch];
            cols.put(slot, child_of(c, level + 1), link_key(i, side), ch);
          } else if (i > 0 && static_cast<uint32_t>(ch - i0) >= static_cast<uint32_t>(T)) {
            // (node 0 is the short-range root: its group grows through the
            // true root's children below, not through its own)
            const uint32_t at = atomicAdd(&s_nout, 1u);
            if (at < kMaxOutside) {
              s_out[at] = ch;
              s_out_slot[at] = static_cast<uint16_t>(slot - static_cast<uint32_t>(slot_0));
            }
          }
        }
      }
      if (MAKE && e[u] > 0) {
        if (up != kNoSlot)
          cols.put_make(up, child_of(code[u], level - e[u] + 1), make_key(i, e[u] - 1),
                        p[u] + e[u] - 1);
        cols.cover(i, p[u], e[u], code[u], level);
      }
    }
    // Chains before the tile that reach into its slots, 64 nodes at a time
    // (P does not decrease and a chain has at most ten slots).
    if (back_wave) {
      int32_t q = back_q, pq = back_p, eq = back_e;
      while (true) {
        if (eq > 0 && pq + eq > cols.base && q >= 1)
          cols.cover(q, pq, eq, b.codes[q], third(b.pn[q]));
        // the earliest node of the 64 starts too early to reach: done
        const int32_t q_min = __builtin_amdgcn_readlane(q, 63);
        const int32_t p_min = __builtin_amdgcn_readlane(pq, 63);
        if (q_min <= 1 || p_min + kMaxEdge <= cols.base) break;
        q -= 64;
        pq = eq = 0;
        if (q >= 1) {
          eq = b.e[q];
          pq = b.p[q];
        }
      }
    }
    if (LINK && i0 == 0 && wave_id() == 1 && b.m >= 1) {
      // The true root's internal children, the nodes whose parent entry is 0:
      // the split of [0, m] (04_radix_tree.cpp:94-104 with d = +1, l = n).
      const uint32_t c0 = b.codes[0];
      const uint32_t dn = delta(c0, b.codes[b.m]);
      const int32_t lane = static_cast<int32_t>(lane_id());
      int32_t lo = 0, hi = b.m;  // the largest x in [lo, hi) above dn; lo is
      while (hi - lo > 1) {
        const int32_t step = (hi - lo + 63) >> 6;
        const int32_t x = lo + step * (lane + 1);
        const int32_t c = __popcll(__ballot(x < hi && delta(c0, b.codes[x]) > dn));
        hi = min(hi, lo + step * (c + 1));
        lo += step * c;
      }
      const int32_t y = lo + lane;
      if (lane < 2 && y >= T && y < b.m) {
        const uint32_t at = atomicAdd(&s_nout, 1u);
        if (at < kMaxOutside) {
          s_out[at] = y;
          s_out_slot[at] = 0;
        }
      }
    }
    __syncthreads();
    if constexpr (LINK) {
      const uint32_t n_out = min(s_nout, static_cast<uint32_t>(kMaxOutside));
      if (static_cast<uint32_t>(tid) < n_out)
        push_subgroup<MAKE>(b, cols, s_out[tid],
                            static_cast<uint32_t>(slot_0) + s_out_slot[tid]);
      __syncthreads();
    }

    // The nodes, a slot per thread, packed over the columns: those of a turn are
    // read before its nodes overwrite them, and a node is shorter than a column.
    // (two calls, not a loop: nearly every tile has one turn, and in a loop 10M
    // points took 166 us, not 162)
    const auto turn = [&](int t) {
      const bool live = t < cols.n;
      int32_t nd[15];
      if (live) {
        const int32_t s = cols.base + t;
        const u64 own = s_owner[t];
        const uint32_t kids = (s_mask[t >> 2] >> ((t & 3) * 8)) & 255u;
        if constexpr (WHOLE) {
#pragma unroll
          for (int c = 0; c < 8; ++c) nd[c] = static_cast<int32_t>(s_child[col_word(t, c)]);
          nd[13] = static_cast<int32_t>(kids);
          nd[14] = 0;
          nd[8] = nd[9] = nd[10] = nd[11] = nd[12] = 0;
        } else {
          __builtin_memcpy(nd, b.nodes + s, sizeof(nd));
          int32_t links = 0;
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const u64 last = s_child[col_word(t, c)];
            const uint32_t key = static_cast<uint32_t>(last >> 32);
            if constexpr (MAKE) {
              // (a zeroed node's word holds at most the key of a chain whose walk
              // left its tile)
              const uint32_t far = static_cast<uint32_t>(nd[c]);
              nd[c] = static_cast<int32_t>(last);
              if (far > key) nd[c] = b.p[(far - 1u) >> 4] + static_cast<int32_t>((far - 1u) & 15u);
              if (far) links |= 1 << c;
            } else if (key) {
              nd[c] = static_cast<int32_t>(last);
              links |= 1 << c;
            }
          }
          if constexpr (MAKE) nd[13] |= links | static_cast<int32_t>(kids);
          else nd[14] &= ~links;
        }
        if (MAKE && (own != 0 || s == 0) && (WHOLE || s != 0)) {
          // Corner and cell size of the chain's step (oct.h:44-57, 76-88); slot
          // 0 is the root of apps/cpu_demo/main.cpp:125-132. Other slots no
          // chain covers stay zero.
          const int32_t lv = s == 0 ? root_level : static_cast<int32_t>((own >> 30) & 15u);
          const uint32_t cd = s == 0 ? b.codes[0] : static_cast<uint32_t>(own) & 0x3fffffffu;
          const uint32_t shift = static_cast<uint32_t>(kMortonBits - 3 * lv) & 31u;
          const uint32_t corner = (cd >> shift) << shift;
          nd[8] = __float_as_int(decode_axis(corner, 0, b.mn, b.rg));
          nd[9] = __float_as_int(decode_axis(corner, 1, b.mn, b.rg));
          nd[10] = __float_as_int(decode_axis(corner, 2, b.mn, b.rg));
          nd[11] = __float_as_int(1.0f);
          const uint32_t sh = static_cast<uint32_t>(lv - root_level) & 31u;
          nd[12] = __float_as_int(b.rg / static_cast<float>(static_cast<int32_t>(1u << sh)));
        }
      }
      __syncthreads();
      if (live) {
#pragma unroll
        for (int c = 0; c < 15; ++c) reinterpret_cast<int32_t*>(s_child)[t * 15 + c] = nd[c];
      }
    };
    static_assert(kCols <= 2 * kThreads, "two turns");
    turn(tid);
    if (cols.n > kThreads) turn(tid + kThreads);
    __syncthreads();
    // Out in whole lines: consecutive lanes store consecutive 16 bytes.
    int32_t* dst = reinterpret_cast<int32_t*>(b.nodes + cols.base);
    const int32_t words = cols.n * 15;
    // (all LDS reads in flight together; those past the last node are not stored)
    constexpr int OUT = (kCols * 15 + kThreads * 4 - 1) / (kThreads * 4);
    constexpr int LAST = kCols * kColWords / 2 - 1;  // in 16 bytes
    v4i x[OUT];
#pragma unroll
    for (int k = 0; k < OUT; ++k)
      x[k] = reinterpret_cast<const v4i*>(s_child)[min(k * kThreads + tid, LAST)];
#pragma unroll
    for (int k = 0; k < OUT; ++k) {
      const int32_t q = (k * kThreads + tid) * 4;
      if (q + 4 <= words) {
        if constexpr (PHASE == kWholeStreamed)
          __builtin_nontemporal_store(static_cast<v4i_any>(x[k]),
                                      reinterpret_cast<v4i_any*>(dst + q));
        else
          __builtin_memcpy(dst + q, &x[k], 16);
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (q + u < words) dst[q + u] = x[k][u];
      }
    }
    __syncthreads();
  }
}

// Before the phase of a per-stage entry: whether the caller's arrays are those
// of a build, as the tiled kernel takes them; *form becomes form_id where they are
// not. (Any other value, an earlier call's among them, means that they are, so the
// word needs no clearing.) A build's are: offsets that are the inclusive scan of
// the counts, counts of at most ten that are the levels between a node and its
// parent, codes of 30 bits that increase, prefix lengths of such codes that grow
// down the tree (or the parent is node 0), and, for the link phase, children and parents that name each
// other, where node 0 stands for the true root. Over repeated codes two nodes of
// one level can be each other's child, and a child be node m.
//
// A tile's nodes find their parents and children in LDS; those with one elsewhere
// are listed and looked up in memory by full waves. What bounds it is the reading
// of every array (link: 23 bytes a node) and its tests. Link of 2M points: 19 us
// when every node gathered its neighbours from memory, 15 with branches between the
// tests (16 with tiles of 1024), 13.
//
// The make call alone has no children arrays to walk down from a slot's owner,
// so the top link of a chain whose walk up leaves its tile comes from below: the
// walk in global memory, and the order key into the child's word of the zeroed
// node, kept by an atomic max, where the scatter of other arrays would put it too.
// The make phase turns it into the link.
constexpr int kCheckTile = 512;
constexpr uint32_t kCheckList = 512;  // of each kind; a build's tile has at most 124 (see 2.)
template <bool LINK>
__global__ __launch_bounds__(kThreads) void check_kernel(OctArgs a) {
  constexpr int T = kCheckTile;
  constexpr int NPT = T / kThreads;
  __shared__ int32_t s_par[T];
  __shared__ uint8_t s_pn[T];
  __shared__ uint8_t s_chain[T];  // make: the count is not 0
  __shared__ uint8_t s_named[T];  // link: by its parent, as a child
  __shared__ uint16_t s_up[kCheckList], s_down[kCheckList];  // nodes; places of children's parents
  __shared__ uint32_t s_n[2];
  const int tid = threadIdx.x;
  const int32_t m = a.n_brt_host;
  const int32_t i0 = static_cast<int32_t>(blockIdx.x) * T;
  // (neighbouring nodes, so that one load takes a thread's)
  const int l0 = tid * NPT;
  const int32_t at0 = i0 + l0;
  int32_t e[NPT], p[NPT], lc[NPT], par[NPT], p_before = 0;
  uint32_t code[NPT], before = 0, next = 0;
  uint8_t pn[NPT], hl[NPT], hr[NPT];
  if (i0 + T <= m) {
    __builtin_memcpy(e, a.edge + at0, sizeof(e));
    __builtin_memcpy(p, a.offsets + at0, sizeof(p));
    __builtin_memcpy(par, a.parent + at0, sizeof(par));
    __builtin_memcpy(code, a.codes + at0, sizeof(code));
    __builtin_memcpy(pn, a.prefix_n + at0, sizeof(pn));
    if constexpr (LINK) {
      __builtin_memcpy(lc, a.left_child + at0, sizeof(lc));
      __builtin_memcpy(hl, a.has_leaf_left + at0, sizeof(hl));
      __builtin_memcpy(hr, a.has_leaf_right + at0, sizeof(hr));
    }
  } else {
#pragma unroll
    for (int u = 0; u < NPT; ++u) {
      const int32_t i = at0 + u;
      e[u] = p[u] = lc[u] = par[u] = 0;
      code[u] = 0;
      pn[u] = hl[u] = hr[u] = 0;
      if (LINK && i == m) code[u] = a.codes[m];
      if (i >= m) continue;
      e[u] = a.edge[i];
      p[u] = a.offsets[i];
      par[u] = a.parent[i];
      code[u] = a.codes[i];
      pn[u] = a.prefix_n[i];
      if constexpr (LINK) {
        lc[u] = a.left_child[i];
        hl[u] = a.has_leaf_left[i];
        hr[u] = a.has_leaf_right[i];
      }
    }
  }
  if (at0 > 0 && at0 < m) {
    p_before = a.offsets[at0 - 1];
    before = a.codes[at0 - 1];
  }
  if (LINK && at0 + NPT <= m) next = a.codes[at0 + NPT];
  const uint32_t pn_0 = a.prefix_n[0];
  uint32_t root = 0;
  if constexpr (LINK) root = delta(a.codes[0], a.codes[m]);
#pragma unroll
  for (int u = 0; u < NPT; ++u) {
    const int l = l0 + u;
    s_par[l] = par[u];
    s_pn[l] = pn[u];
    if constexpr (LINK) s_named[l] = 0;
    else s_chain[l] = e[u] != 0;
  }
  if (tid < 2) s_n[tid] = 0;
  __syncthreads();
  const auto in_tile = [&](int32_t q) { return static_cast<uint32_t>(q - i0) < static_cast<uint32_t>(T); };
  const auto is_node = [&](int32_t q) { return static_cast<uint32_t>(q) < static_cast<uint32_t>(m); };
  // (all tests of a node without branches: its few loads and LDS reads are bounded
  // by selects, and most of what this kernel takes is instructions)
  bool bad = false;
  // (a full list: not a build's)
  const auto push = [&](uint16_t* list, int which, uint32_t l) {
    const uint32_t at = atomicAdd(&s_n[which], 1u);
    if (at < kCheckList) list[at] = static_cast<uint16_t>(l);
    else bad = true;
  };
#pragma unroll
  for (int u = 0; u < NPT; ++u) {
    const int32_t i = at0 + u;
    const uint32_t l = static_cast<uint32_t>(l0 + u);
    const uint32_t code_l = u ? code[u - 1] : before, code_r = u + 1 < NPT ? code[u + 1] : next;
    const bool live = i < m, inner = live & (i != 0);
    const int32_t up = par[u];
    bad |= live & ((code[u] >= kCodeEnd) | (pn[u] > kMaxPrefix));
    if constexpr (LINK) bad |= live & ((code[u] >= code_r) | (code_r >= kCodeEnd) | !is_node(lc[u]));
    bad |= live & (i == 0) & ((e[u] | p[u]) != 0);
    bad |= inner & ((static_cast<uint32_t>(e[u]) > static_cast<uint32_t>(kMaxEdge)) |
                    (static_cast<uint32_t>(p[u]) - static_cast<uint32_t>(u ? p[u - 1] : p_before) !=
                     static_cast<uint32_t>(e[u])) |
                    (code_l >= code[u]) | !is_node(up));
    const bool near = (up == 0) | in_tile(up);
    const uint32_t own = pn[u];
    const uint32_t pn_up = up == 0 ? pn_0 : s_pn[in_tile(up) ? up - i0 : 0];
    bad |= inner & near &
           ((third(own) - third(pn_up) != e[u]) | (pn_up > kMaxPrefix) |
            ((up != 0) & (pn_up >= own)));
    if (inner & !near & is_node(up)) push(s_up, 0, l);
    if constexpr (LINK) {
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        const bool inside = inner & ((side == 0 ? hl[u] : hr[u]) == 0);
        const int32_t ch = lc[u] + side;
        const bool node = is_node(ch) & (ch != 0), here = in_tile(ch);
        const bool named = s_par[here ? ch - i0 : 0] == i;
        bad |= inside & (!node | (here & !named));
        if (inside & here & named) s_named[ch - i0] = 1;
        if (inside & node & !here) push(s_down, 1, l * 2u + static_cast<uint32_t>(side));
      }
      // The true root's children lie on either side of the pair of codes with the
      // shortest common prefix.
      const bool of_root = (delta(code[u], code_r) == root) | (delta(code_l, code[u]) == root);
      bad |= inner & (of_root != (up == 0));
    } else if (inner & (e[u] > 0) & is_node(up)) {
      bool far = false;  // out of the octree kernel's tile: the numbers differ above its bits
      int32_t h = up;
      for (int hop = 0; hop < 31; ++hop) {
        far |= (h ^ i) >= kOctTile;
        if (!in_tile(h) || s_chain[h - i0] != 0) break;
        const int32_t next_up = s_par[h - i0];
        if (next_up == h) break;
        h = next_up;
      }
      if (far) push(s_down, 1, l);
    }
  }
  __syncthreads();
  if constexpr (LINK) {
    // (a parent in the tile has named its children there)
#pragma unroll
    for (int u = 0; u < NPT; ++u)
      bad |= (at0 + u < m) & (at0 + u > 0) & (par[u] != 0) & in_tile(par[u]) &
             (s_named[l0 + u] == 0);
  }
  for (uint32_t q = tid; q < min(s_n[0], kCheckList); q += kThreads) {
    const uint32_t l = s_up[q];
    const int32_t i = i0 + static_cast<int32_t>(l), up = s_par[l];
    const uint32_t own = s_pn[l], pn_up = a.prefix_n[up];
    bad |= (third(own) - third(pn_up) != a.edge[i]) | (pn_up >= own);
    if constexpr (LINK) {
      const int32_t at = a.left_child[up];
      const bool leaf_l = a.has_leaf_left[up], leaf_r = a.has_leaf_right[up];
      bad |= !(i == at ? !leaf_l : (i == at + 1) & !leaf_r);
    }
  }
  for (uint32_t q = tid; q < min(s_n[1], kCheckList); q += kThreads) {
    const uint32_t l = s_down[q];
    if constexpr (LINK) {
      const int32_t i = i0 + static_cast<int32_t>(l >> 1);
      bad |= a.parent[a.left_child[i] + static_cast<int32_t>(l & 1u)] != i;
    } else {
      const int32_t i = i0 + static_cast<int32_t>(l);
      const int32_t n_new = a.edge[i];
      put_word(a, a.offsets[make_head(a, i)], child_of(a.codes[i], s_pn[l] / 3 - n_new + 1),
               make_key(i, n_new - 1));
    }
  }
  if (bad) *a.form = a.form_id;
}

// After a scatter of order keys: the keys of the slots of chain i become the
// values that they stand for, and a make call's slots get their corner and cell
// size. Chain i owns slot P[i]+j when no later chain covers it; every slot that
// receives a child write is covered by a chain or is the root slot 0.
template <bool MAKE>
__device__ __forceinline__ void resolve_children(const OctArgs& a, int32_t slot) {
  int32_t* ch = a.nodes[slot].children;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const uint32_t v = static_cast<uint32_t>(ch[c]);
    if (v == 0 || (v >> 31) == (MAKE ? 1u : 0u)) continue;
    if constexpr (MAKE) {
      // (a chain of more than 16 steps, over codes that differ in bit 31, can run
      // into the next numbers: nothing is read past the arrays)
      const uint32_t i = (v - 1u) >> 4;
      if (i < static_cast<uint32_t>(a.n_brt_host))
        ch[c] = a.offsets[i] + static_cast<int32_t>((v - 1u) & 15u);
    } else {
      const uint32_t q = v & 0x7fffffffu;
      ch[c] = a.left_child[q >> 1] + static_cast<int32_t>(q & 1u);
    }
  }
}
template <bool MAKE>
__global__ __launch_bounds__(256) void resolve_kernel(OctArgs a, float mn, float rg) {
  if (*a.form != a.form_id) return;
  const int32_t m = a.n_brt_host;
  for (int32_t i = blockIdx.x * 256 + static_cast<int32_t>(threadIdx.x); i < m;
       i += static_cast<int32_t>(gridDim.x) * 256) {
    if (i == 0) {
      resolve_children<MAKE>(a, 0);
      continue;
    }
    const int32_t e = a.edge[i];
    if (e <= 0) continue;
    const int32_t p = a.offsets[i];
    const int32_t last = p + e - 1;
    uint32_t owned = e >= 32 ? ~0u : (1u << e) - 1u;
    for (int32_t k = i + 1; k < m && owned; ++k) {
      const int32_t pk = a.offsets[k];
      if (pk > last) break;
      const int32_t ek = a.edge[k];
      if (ek <= 0) continue;
      const int32_t lo = max(pk, p) - p, hi = min(pk + ek - 1, last) - p;
      for (int32_t q = lo; q <= min(hi, 31); ++q) owned &= ~(1u << q);
    }
    const int32_t root_level = a.prefix_n[0] / 3, level = a.prefix_n[i] / 3;
    const uint32_t code = a.codes[i];
    for (int32_t j = 0; j < e && j < 32; ++j) {
      const int32_t slot = p + j;
      // (slot 0 is the root's)
      if (!((owned >> j) & 1u) || slot <= 0 || slot >= a.k_host) continue;
      if constexpr (MAKE) {
        OctNode* nd = a.nodes + slot;
        const uint32_t shift = static_cast<uint32_t>(kMortonBits - 3 * (level - j)) & 31u;
        const uint32_t corner = (code >> shift) << shift;
        nd->corner[0] = decode_axis(corner, 0, mn, rg);
        nd->corner[1] = decode_axis(corner, 1, mn, rg);
        nd->corner[2] = decode_axis(corner, 2, mn, rg);
        nd->corner[3] = 1.0f;
        const uint32_t sh = static_cast<uint32_t>(level - j - root_level) & 31u;
        nd->cell_size = rg / static_cast<float>(static_cast<int32_t>(1u << sh));
      }
      resolve_children<MAKE>(a, slot);
    }
  }
}

// Root node of apps/cpu_demo/main.cpp:125-132 alone (the per-stage entry
// point that stands in for that host code).
__global__ void oct_root_kernel(OctNode* nodes, const uint32_t* codes,
                                const uint8_t* prefix_n, int32_t n_brt,
                                float mn, float rg) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const int32_t root_level = n_brt >= 1 ? prefix_n[0] / 3 : 0;
  const uint32_t shift = static_cast<uint32_t>(kMortonBits - 3 * root_level) & 31u;
  const uint32_t c = (codes[0] >> shift) << shift;
  nodes->corner[0] = decode_axis(c, 0, mn, rg);
  nodes->corner[1] = decode_axis(c, 1, mn, rg);
  nodes->corner[2] = decode_axis(c, 2, mn, rg);
  nodes->corner[3] = 1.0f;
  nodes->cell_size = rg;
}

}  // namespace

void launch_oct_root(OctNode* nodes, const uint32_t* codes,
                     const uint8_t* prefix_n, int32_t n_brt, float mn,
                     float rg, hipStream_t s) {
  oct_root_kernel<<<1, 64, 0, s>>>(nodes, codes, prefix_n, n_brt, mn, rg);
}

bool launch_oct_build(const OctArgs& a, const SegView& sv, const int32_t* tile_start,
                      int32_t total_tiles, const OctSingle& single, hipStream_t s) {
  // The pushes read every array of the radix tree; the per-segment counts,
  // node bases and the fit flag come from the build.
  if (!a.has_leaf_left || !a.has_leaf_right || !a.left_child || !a.parent || !a.codes ||
      !a.prefix_n || !a.edge || !a.offsets || !a.nodes || !a.ctrl || !a.n_unique ||
      !a.oct_start || !a.kalloc)
    return false;
  if (total_tiles <= 0) return true;
  if (single.mail && (sv.n_seg != 1 || !single.oct_start || !single.ctrl)) return false;
  const auto go = [&](auto kernel) {
    kernel<<<total_tiles, kThreads, 0, s>>>(a, sv, tile_start, single);
  };
  if (single.mail && a.stream_nodes) go(oct_build_kernel<true, kWholeStreamed>);
  else if (single.mail) go(oct_build_kernel<true, kWhole>);
  else if (a.stream_nodes) go(oct_build_kernel<false, kWholeStreamed>);
  else go(oct_build_kernel<false, kWhole>);
  return true;
}

namespace {
// (a grid that fills the chip; it returns at once for a build's arrays)
template <bool MAKE>
void launch_resolve(const OctArgs& a, const SegView& sv, hipStream_t s) {
  const int32_t blocks = (a.n_brt_host + 255) / 256;
  resolve_kernel<MAKE><<<blocks < 2048 ? blocks : 2048, 256, 0, s>>>(a, sv.min1, sv.range1);
}
}  // namespace

void launch_oct_make(const OctArgs& a, const SegView& sv, hipStream_t s) {
  check_kernel<false><<<(a.n_brt_host + kCheckTile - 1) / kCheckTile, kThreads, 0, s>>>(a);
  oct_build_kernel<false, kMakePhase>
      <<<(a.n_brt_host + kOctTile - 1) / kOctTile, kThreads, 0, s>>>(a, sv, nullptr, OctSingle{});
  launch_resolve<true>(a, sv, s);
}

void launch_oct_link(const OctArgs& a, const SegView& sv, hipStream_t s) {
  check_kernel<true><<<(a.n_brt_host + kCheckTile - 1) / kCheckTile, kThreads, 0, s>>>(a);
  oct_build_kernel<false, kLinkPhase>
      <<<(a.n_brt_host + kOctTile - 1) / kOctTile, kThreads, 0, s>>>(a, sv, nullptr, OctSingle{});
  launch_resolve<false>(a, sv, s);
}

}  // namespace ocp
