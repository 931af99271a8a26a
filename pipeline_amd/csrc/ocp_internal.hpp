// Host-side launchers of the stage kernels (one translation unit per stage)
// and the shared control block. Every launcher is asynchronous on `stream`
// and takes device pointers only.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ocp_device.hpp"

namespace ocp {

// Control words in device memory (one block per context).
enum CtrlSlot : int {
  // words 0-7 are unused (tiles take their index from the workgroup id)
  kCtrlEpoch = 8,      // bumped once per launch group; tags lookback flags
  kCtrlOctTotal = 9,   // total octree slots of the batch
  kCtrlOctOk = 10,     // 1 when the octree fits the node capacity
  kCtrlMsdBig = 11,    // MSD sort: digits listed for the second level,
  kCtrlLearnBad = 12,  // learned sort: misordered bucket boundaries
  kCtrlTimeout = 13,   // mark of the launch whose wait gave up (0: none)
  kCtrlWaitLimit = 14, // 0: waits poll up to kSpinLimit times; v > 0: v - 1
  kCtrlMsdTiles = 15,  // ... their tiles
  kCtrlMsdSlots = 16,  // ... and the count slots of their long runs
  kCtrlOctForm = 17,   // last make or link call whose arrays were not a build's
  kCtrlMailAt = 18,    // (two words) where the host reads of a time-out
  kCtrlWords = 64,
};

// Polls a bounded wait may spend before it gives up (set from the host with
// ocp_set_wait_limit; 0 makes every wait give up at once).
__device__ __forceinline__ uint32_t wait_limit(const uint32_t* ctrl) {
  const uint32_t v = ctrl[kCtrlWaitLimit];
  return v ? v - 1u : kSpinLimit;
}

// A wait that gives up stores its launch's mark (below) in kCtrlTimeout;
// the first one wins, later ones store the same mark. The keys such a pass
// leaves may no longer match the digit counts the next pass is sized by, so
// every later kernel that consumes lookback output does nothing until the
// host has reported the error and cleared the word. A kernel stops only on
// the mark of an earlier launch: that value cannot change while it runs
// (tiles of the running launch can only store its own mark), so every
// thread of every workgroup takes the same branch.
__device__ __forceinline__ uint32_t timeout_mark(uint32_t tag) { return tag | 0x80000000u; }
__device__ __forceinline__ bool stopped(const uint32_t* ctrl, uint32_t tag) {
  const uint32_t v = ctrl[kCtrlTimeout];
  return v != 0u && v != timeout_mark(tag);
}
// The host's own word is told as well: what it last heard of a build would not
// show the time-out of a launch replayed from a caller's graph since.
__device__ __forceinline__ void raise_timeout(uint32_t* ctrl, uint32_t tag) {
  ctrl[kCtrlTimeout] = timeout_mark(tag);
  const uint64_t at = *reinterpret_cast<const uint64_t*>(ctrl + kCtrlMailAt);
  __hip_atomic_store(reinterpret_cast<uint32_t*>(at), timeout_mark(tag), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}
// Kernels without waits stop on any mark.
__device__ __forceinline__ bool stopped_any(const uint32_t* ctrl) {
  return ctrl[kCtrlTimeout] != 0u;
}

// Lookback stage ids (part of every flag tag).
enum Stage : uint32_t {
  kStagePass0 = 0,  // OneSweep passes 0..3
  kStageUnique = 4,
  kStageScan = 5,
  kStageBucket = 6,  // learned sort: 6 and 7
};

// Kernel configuration chosen by the autotuner (or the defaults).
struct TuneTable {
  int sort_waves = 8;      // OneSweep workgroup = sort_waves * 64 threads
  int sort_kpt = 16;       // keys per thread in OneSweep
  int morton_ppt = 16;     // points per thread in the Morton kernel
  int morton_grid = 1024;  // persistent Morton workgroups
  int scan_ipt = 16;       // items per thread in unique / edge-scan tiles
  int sort_bits = 8;       // digit width of a build's sort: 8 (4 passes) or 10 (3)
  int sort10_kpt = 8;      // keys per thread of a 10-bit pass (16 waves)
  int oct_order = 0;       // 0 or 1, kept for saved tables: one octree kernel serves both
  int sort_msd = 0;        // 10-bit digits: LSD passes (0) or MSD scatter + LDS windows (1)
};

inline int sort_tile(const TuneTable& t) { return t.sort_waves * 64 * t.sort_kpt; }
// Digit width of a build's sort passes: 10-bit digits (three passes over
// the 30-bit Morton keys) when chosen and no permutation rides along.
inline int pipe_sort_bits(const TuneTable& t, bool perm) {
  return (t.sort_bits == 10 && !perm) ? 10 : 8;
}
// The MSD form: chosen, 10-bit digits, and few enough segments that 1024
// counts and cursors each are no more than the keys.
constexpr int32_t kMsdMaxSegments = 2048;
inline bool pipe_sort_msd(const TuneTable& t, bool perm, int32_t n_seg) {
  return t.sort_msd != 0 && pipe_sort_bits(t, perm) == 10 && n_seg <= kMsdMaxSegments;
}
// A build whose caller set no table takes the MSD form by itself, unless it
// carries the permutation (its passes are stable) or has more clouds than that
// form takes. Whole builds, four 8-bit passes against it, uniform points:
// 307,200 114 -> 92 us, 2^20 150 -> 120, 2^22 322 -> 240, 10M 596 -> 475.
// Below 16,384 points the sort is launches either way.
inline bool auto_sort_msd(int64_t n, int32_t n_seg, bool perm) {
  return !perm && n >= 16384 && n_seg <= kMsdMaxSegments;
}
// Where many keys crowd into few digits, most of them take the second level:
// 2^24 clustered points 528 -> 495 us, but 2^20 133 -> 147 and 10M 315 -> 341.
// So below 12M points a cloud, a build after which more than a sixteenth of the
// keys turns out to have gone there (the host learns it with the counts) is
// followed by kSkewBuilds builds of about its size with LSD passes, then by
// another try. The result is the same either way.
inline bool auto_sort_skew(int64_t max_seg) { return max_seg < 12000000; }
constexpr int32_t kSkewBuilds = 256;
// Those passes' digits, for one cloud: three passes of 10 bits while the tiles'
// 1024 runs stay in the caches, else four of 8. Clustered points, four passes
// against three: 307,200 105 -> 98 us, 2^20 133 -> 126, 2^21 166 -> 151, but 2^22
// 208 -> 212 and 10M 315 -> 347.
inline bool crowd_sort10(int64_t n, int32_t n_seg) { return n_seg <= 1 && n < 3000000; }
// Tiles of 16K keys for the scatter once there are enough of them (10M: 47 ->
// 39 us), else of 8K.
inline int auto_sort10_kpt(int64_t max_seg) { return max_seg >= (int64_t(1) << 22) ? 16 : 8; }
inline int pipe_sort_tile(const TuneTable& t, bool perm) {
  return pipe_sort_bits(t, perm) == 10 ? 1024 * t.sort10_kpt : sort_tile(t);
}
// Digit-count words per segment: four 256-bin histograms for 8-bit digits,
// three 1024-bin ones for 10-bit digits.
constexpr int hist_stride(int bits) { return bits == 10 ? 3 * 1024 : 4 * 256; }
inline int morton_tile(const TuneTable& t) { return 256 * t.morton_ppt; }
inline int scan_tile(const TuneTable& t) { return 256 * t.scan_ipt; }
constexpr int kNodeTile = 256;  // BRT nodes per tile of the per-stage radix tree
constexpr int kOctTile = 512;   // ... of the octree kernel

bool sort_config_supported(int waves, int kpt);
bool sort10_config_supported(int kpt);
bool scan_config_supported(int ipt);
bool morton_config_supported(int ppt);

// ---- utility kernels (k_util.hip)
// bytes must be a multiple of 16 and both pointers 16-byte aligned.
void launch_copy(void* dst, const void* src, int64_t bytes, hipStream_t s);
struct Affine {
  float m[12];  // rows of A (3x3), then t
};
void launch_transform(const float* src, float* dst, int64_t n, bool float3, const Affine& m,
                      float lo, float hi, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t value, int64_t n_words,
                     hipStream_t s);
// Bump the epoch and clear the learned sort's misorder count; optionally
// zero n_hist words of histogram and n2 words at z2.
void launch_begin(uint32_t* ctrl, uint32_t* hist, int64_t n_hist,
                  hipStream_t s, uint32_t* z2 = nullptr, int64_t n2 = 0);
// Begin for lookback flags shared by every context on the device: the new
// epoch is past both the context's and *dev_epoch, and is stored in both.
void launch_begin_shared(uint32_t* ctrl, uint32_t* dev_epoch, uint32_t* hist, int64_t n_hist,
                         hipStream_t s);
// mail (pinned host memory): the build's time-out mark, slot total and fit
// flag at their control-word places, then, for at most kMailSegs segments, the
// counts n_unique and kalloc kMailSegs words apart.
constexpr int32_t kMailSegs = 4096;
constexpr int32_t kMailWords = kCtrlWords + 2 * kMailSegs;
void launch_oct_offsets(const int32_t* n_unique, const int32_t* kalloc, int32_t n_seg,
                        int32_t* oct_start, uint32_t* ctrl, int64_t k_cap, uint32_t* mail,
                        hipStream_t s);
void launch_zero_nodes(OctNode* nodes, const uint32_t* ctrl, int64_t k_cap,
                       hipStream_t s);

// ---- input side (k_init.hip)
// n float4 points from the reference's hybrid Tausworthe generator.
void launch_init_random(float* out, int32_t n, float mn, float rg, int32_t seed, hipStream_t s);
// Per-segment cube boxes into mn[n_seg], rg[n_seg]; mm: 2 * n_seg words of
// scratch. Tiles of `tile` points per the tile map.
void launch_boxes(const float* pts, bool float3, const SegView& sv, const int32_t* tile_start,
                  int32_t total_tiles, int tile, uint32_t* mm, float* mn, float* rg,
                  hipStream_t s);

// ---- stage 1 (k_morton.hip)
// hist (optional): per-segment digit counts of the keys for hist_bits-wide
// digits (8: four 256-bin histograms; 10: three 1024-bin ones; kHistTop10:
// only the third of those, the top 10-bit digit, in the same layout).
constexpr int kHistTop10 = 1;
void launch_morton(const float* pts, bool float3, uint32_t* keys,
                   const SegView& sv, const int32_t* tile_start,
                   int32_t total_tiles, uint32_t* hist, const TuneTable& tt,
                   hipStream_t s, int hist_bits = 8);

// ---- stage 2 (k_onesweep.hip)
void launch_histogram(const uint32_t* keys, const SegView& sv,
                      const int32_t* tile_start, int32_t total_tiles,
                      uint32_t* hist, const TuneTable& tt, hipStream_t s);
// Same, over tiles of `tile` keys (a tile map built for another tile size).
void launch_histogram_tiles(const uint32_t* keys, const SegView& sv,
                            const int32_t* tile_start, int32_t total_tiles,
                            int tile, uint32_t* hist, const TuneTable& tt,
                            hipStream_t s, uint32_t* cursor0 = nullptr);
// (cursor0, optional: n_seg * 256 words zeroed for launch_cursor_pass0)
// stable = false: equal digits may leave in any order (the first pass of a
// sort of bare keys); full tiles then rank with LDS atomics. bits = 10: the
// pass takes 10-bit digits (16-wave tiles of 1024 * sort10_kpt keys, 1024
// flags per tile, hist laid out for 10-bit digits).
void launch_onesweep_pass(const uint32_t* in, uint32_t* out,
                          const SegView& sv, const int32_t* tile_start,
                          int32_t total_tiles, const uint32_t* hist,
                          uint64_t* flags, uint32_t* ctrl, int pass, bool stable,
                          const TuneTable& tt, hipStream_t s, int bits = 8);
// MSD sort of bare 30-bit keys (k_msd.hip): the scatter by the top 10-bit
// digit (histogram slot 2 of the 10-bit histograms) without a lookback (cursor
// holds n_seg * 1024 zeroed words, claimed by atomic adds; tiles of 1024 *
// sort10_kpt keys), LDS sorts of windows of msd_window(...) keys of the
// result, and a second level for the digits too large for LDS.
struct MsdLevel2 {
  int4* big;         // listed digits {first key, keys, top digit, first shared slot}
  int2* tiles;       // second-level tiles {listed digit, tile in it}
  uint32_t* hist;    // [max_big][1024] counts of bits 10-19
  uint32_t* cursor;  // [max_big][1024]
  uint32_t* hist3;   // [max_slots][1024] low-bit counts of long one-prefix runs
  int32_t max_big, max_tiles, max_slots;
};
// Segments of up to 2800 keys a digit on average sort windows in 4096-key
// workgroups of four waves (four a CU by LDS), larger ones in 12288-key
// workgroups of eight (two a CU): at 2^20 points 1024 keys a digit, 10M 9800.
inline bool msd_small(int64_t max_seg) { return max_seg <= 1024 * 2800; }
// Keys per window of a segment of len keys; 0: one workgroup per digit, where a
// digit about fills it. By the segment, not the batch's largest: with the latter a
// batch of one cloud of 6.2M points and 2000 of 100 launched two million
// workgroups (7,970 us a build, now 352).
__host__ __device__ inline int32_t msd_window(bool small, int64_t len) {
  return small ? 1024 : len <= 1024 * 6000 ? 4096 : 0;
}
inline int64_t msd_windows(int64_t len, int64_t max_seg) {
  const int32_t w = msd_window(msd_small(max_seg), len);
  return w ? (len + w - 1) / w : 1024;
}
// Room for the second level of n keys, whatever they are: listed digits hold
// more than the LDS capacity each.
inline void msd_level2_caps(int64_t n, int64_t max_seg, MsdLevel2* l2) {
  l2->max_big = static_cast<int32_t>(n / (msd_small(max_seg) ? 4096 : 12288) + 1);
  l2->max_tiles = static_cast<int32_t>(n / 8192 + l2->max_big + 1);
  l2->max_slots = static_cast<int32_t>(n / 65536 + 1);
}
void launch_msd_scatter(const uint32_t* in, uint32_t* out, const SegView& sv,
                        const int32_t* tile_start, int32_t total_tiles, const uint32_t* hist,
                        uint32_t* cursor, const uint32_t* ctrl, const TuneTable& tt,
                        hipStream_t s);
void launch_msd_windows(uint32_t* keys, const SegView& sv, const int32_t* tile_start,
                        int32_t total_tiles, int64_t max_seg, const uint32_t* hist,
                        const MsdLevel2& l2, uint32_t* ctrl, hipStream_t s);
// `other` is overwritten where digits are listed. The grids are what n keys of
// segments of at most max_seg can need, however much room l2 has by now.
void launch_msd_level2(uint32_t* keys, uint32_t* other, const MsdLevel2& l2, int64_t n,
                       int64_t max_seg, const uint32_t* ctrl, hipStream_t s);
// Cursor words per segment after the segments' histograms (the first sort
// pass's or the MSD scatter's: one per digit, at most 1024).
constexpr int kCursorWords = 1024;
// First pass of an LSD sort of bare keys (digit key & 255, or key & 1023
// with bits == 10; any order among equal digits) as a cursor scatter
// (cursor_scatter.hpp): no lookback; one zeroed cursor per segment and
// digit (n_seg * 2^bits words); hist as the OneSweep passes read it (slot
// 0); tiles as OneSweep's of the tile table.
void launch_cursor_pass0(const uint32_t* in, uint32_t* out, const SegView& sv,
                         const int32_t* tile_start, const int32_t* tiles_dev, int32_t grid,
                         const uint32_t* hist, uint32_t* cursor, const uint32_t* ctrl,
                         const TuneTable& tt, hipStream_t s, int bits = 8);

// Stable pass carrying a value with every key (vin == nullptr: the key's
// index in its segment).
void launch_onesweep_pass_kv(const uint32_t* in, uint32_t* out, const uint32_t* vin,
                             uint32_t* vout, const SegView& sv, const int32_t* tile_start,
                             int32_t total_tiles, const uint32_t* hist, uint64_t* flags,
                             uint32_t* ctrl, int pass, const TuneTable& tt, hipStream_t s);

// ---- stage 3 (k_unique.hip)
// vin/vout (optional): each kept key's value (the first of its run) is
// compacted beside it.
void launch_unique(const uint32_t* in, uint32_t* out, const SegView& sv,
                   const int32_t* tile_start, int32_t total_tiles,
                   uint64_t* flags, uint32_t* ctrl, int32_t* n_unique,
                   int32_t* kalloc, const TuneTable& tt, hipStream_t s,
                   const uint32_t* vin = nullptr, uint32_t* vout = nullptr);

// ---- stage 4 (k_radix_tree.hip)
// The per-stage entry: n nodes over n + 1 sorted codes of any value.
// ctrl (optional): the kernel does nothing once a lookback wait gave up.
void launch_radix_tree(const uint32_t* codes, uint8_t* prefix_n, uint8_t* has_leaf_left,
                       uint8_t* has_leaf_right, int32_t* left_child, int32_t* parent, int32_t n,
                       const uint32_t* ctrl, hipStream_t s);
// The fused build: segments of strictly increasing 30-bit codes, n_unique[k]
// of them in segment k; writes the edge counts of stage 5 as well. Tiles of
// `tile` = tree_tile(...) nodes per the tile map.
void launch_radix_pairs(const uint32_t* codes, uint8_t* prefix_n, uint8_t* has_leaf_left,
                        uint8_t* has_leaf_right, int32_t* left_child, int32_t* parent,
                        int32_t* edge, const SegView& sv, const int32_t* tile_start,
                        int32_t total_tiles, int tile, const int32_t* n_unique,
                        const uint32_t* ctrl, hipStream_t s);
// Nodes per tile of launch_radix_pairs for a build of n points: 2048 once
// that still gives every CU several workgroups (10M points, before the listed
// search: 66 us against 74 with 512), 512 below (2^20 points: 16.4 us against
// 19.6).
inline int tree_tile(int64_t n) { return n >= (int64_t(1) << 21) ? 2048 : 512; }

// ---- stages 5 + 6 (k_edge_scan.hip)
// Edge count of one segment of n nodes (the per-stage entry).
void launch_edge_count(const uint8_t* prefix_n, const int32_t* parent, int32_t* edge, int32_t n,
                       const uint32_t* ctrl, hipStream_t s);
// Inclusive scan of `edge` per segment, one lookback chain each. With
// n_unique, segment k has n_unique[k] - 1 entries and its octree slot count,
// max(1, max P[i] + e[i]), is folded into kalloc[k]; else n_host entries.
void launch_edge_scan(const int32_t* edge, int32_t* offsets, const SegView& sv,
                      const int32_t* tile_start, int32_t total_tiles, const int32_t* n_unique,
                      int32_t n_host, uint64_t* flags, uint32_t* ctrl, int32_t* kalloc,
                      const TuneTable& tt, hipStream_t s);

// ---- stages 1 to 6 of small clouds (k_small.hip), one workgroup each: every
// output of those stages at the segments' point offsets.
constexpr int64_t kSmallCloud = 8192;
// Up to here because 8192 points' keys, sort and tree take 147 KB of the 160 KB of
// LDS; up to there the kernel is the faster one for one cloud (8192 clustered
// points 63 us to the general path's 100) as for batches of any length
// (k_small.hip). Builds with point indices sort pairs, a table other than the
// default and stage timing name the stages' kernels: these keep the general path.
inline bool small_clouds(int64_t max_seg, int32_t n_seg, bool perm) {
  return !perm && max_seg <= kSmallCloud && n_seg >= 1;
}
struct SmallOut {
  uint32_t* sorted;
  uint32_t* unique;
  uint8_t* prefix;
  uint8_t* hl;
  uint8_t* hr;
  int32_t* lc;
  int32_t* par;
  int32_t* edge;
  int32_t* offs;
  int32_t* n_unique;
  int32_t* kalloc;
};
void launch_small_clouds(const float* pts, bool float3, const SegView& sv, int64_t max_seg,
                         bool device_boxes, float* box_min, float* box_range, const SmallOut& o,
                         uint32_t* ctrl, hipStream_t s);

// Sort of at most kSmallSort keys in place by one workgroup: what LDS holds, and
// up to there faster than the six launches of the passes, for spread keys (2000:
// 41 -> 8 us, 16,384: 46 -> 19) as for those that take its radix passes (16,384
// clustered ones 46 -> 36, of a few values in the top bits 44 -> 41).
constexpr uint32_t kSmallSort = 16384;
void launch_small_sort(uint32_t* keys, int32_t n, const uint32_t* ctrl, hipStream_t s);

// ---- stage 7 (k_octree.hip)
struct OctArgs {
  OctNode* nodes;            // base of all segments' nodes
  const int32_t* oct_start;  // per-segment node base (nullptr: 0)
  const int32_t* kalloc;     // per-segment slot count (nullptr: k_host)
  int32_t k_host;
  const uint32_t* ctrl;      // kCtrlOctOk checked when non-null
  const uint32_t* codes;
  const uint8_t* prefix_n;
  const uint8_t* has_leaf_left;
  const uint8_t* has_leaf_right;
  const int32_t* left_child;
  const int32_t* parent;
  const int32_t* edge;
  const int32_t* offsets;
  const int32_t* n_unique;  // per segment (nullptr: n_brt_host + 1)
  int32_t n_brt_host;
  bool stream_nodes;  // nodes past the caches (oct_stream)
  // Per-stage entries: *form == form_id once a kernel of this call has found
  // arrays that are not a build's.
  uint32_t* form;
  uint32_t form_id;
};
// Whether a build of n points stores its nodes past the caches: once they and
// the arrays they are made from outgrow the 256 MB behind the L2s, where they
// only push out what is still to be read (octree of 10M points 151 -> 135 us,
// builds of 8M 335 -> 303, of 4M 207 -> 203); nodes of smaller builds are still
// there for whoever reads them next (compact form of 1M points 35 us, 40 when
// they are not).
inline bool oct_stream(int64_t n) { return n >= (int64_t(1) << 22); }
void launch_oct_root(OctNode* nodes, const uint32_t* codes,
                     const uint8_t* prefix_n, int32_t n_brt, float mn,
                     float rg, hipStream_t s);
// The fused make + link + root pass: writes every slot, zero gaps included.
// Needs every OctArgs array (the fused build has them all); returns false
// (and launches nothing) when an array it needs is null.
// single (one segment with points): the kernel does the offsets kernel's work
// as well, which there is two comparisons. Eight frames of 1M points in a stream
// 715 -> 680 us without that launch, 307,200 points 85 -> 81, 6M 287 -> 283; 10M
// points took 437 us with it and 439 without, so from 2^23 on it is launched.
inline bool oct_single(int64_t n) { return n < (int64_t(1) << 23); }
struct OctSingle {
  int32_t* oct_start;
  uint32_t* ctrl;
  uint32_t* mail;  // null: the offsets kernel has run
  uint32_t k_cap;
};
bool launch_oct_build(const OctArgs& a, const SegView& sv, const int32_t* tile_start,
                      int32_t total_tiles, const OctSingle& single, hipStream_t s);

// The per-stage entries: the make writes (without the children arrays, which may
// be null) or the link writes of n_brt_host nodes, into the k_host nodes that the
// caller prepared. The same kernel where the arrays have a build's form, which a
// kernel before it checks; else a scatter and a kernel that resolves it.
void launch_oct_make(const OctArgs& a, const SegView& sv, hipStream_t s);
void launch_oct_link(const OctArgs& a, const SegView& sv, hipStream_t s);

// ---- node formats and validator (k_format.hip). Node counts come from
// oct_start[n_seg] on the device; boxes are per segment (smin/srg) or the
// scalars mn1/rg1.
constexpr int kTreeReportFields = 12;
void launch_seg_roots(const uint32_t* codes, const uint8_t* prefix_n, const int32_t* n_unique,
                      const int32_t* seg_start, int32_t n_seg, int32_t* root_level,
                      uint32_t* root_code, hipStream_t s);
// cov: one byte per slot, zeroed; rep: kTreeReportFields counters, zeroed.
void launch_validate(const OctNode* nodes, const int32_t* edge, const int32_t* offs,
                     const int32_t* n_unique, const int32_t* oct_start, const int32_t* seg_start,
                     int32_t n_seg, const float* smin, const float* srg, float mn1, float rg1,
                     const int32_t* root_level, const uint32_t* root_code, uint8_t* cov,
                     unsigned long long* rep, hipStream_t s);
// What the compact form is made from: k_total slots of a build.
struct CompactSource {
  const OctNode* nodes;
  int64_t k_total;
  const int32_t* oct_start;
  int32_t n_seg;
  const float* smin;
  const float* srg;
  float mn1, rg1;
  const int32_t* seg_start;
  const int32_t* n_unique;
  const uint8_t* prefix_n;
};
int64_t compact_tiles(int64_t k_total);
// In one pass, in the lookback epoch that a launch_begin before it began (flags:
// 2 * compact_tiles(k_total) words; *bad zeroed). out and children may be null.
// mail: three words of host memory, zeroed (see compact_kernel).
void launch_compact(const CompactSource& c, uint64_t* flags, uint32_t* ctrl, void* out,
                    int32_t* children, int64_t child_cap, unsigned long long* bad, uint32_t* mail,
                    hipStream_t s);
// In two, without waits between workgroups (words: compact_words(k_total)); with
// out null the sizes only.
int64_t compact_words(int64_t k_total);
void launch_compact_no_wait(const CompactSource& c, uint32_t* words, void* out, int32_t* children,
                            int64_t child_cap, uint32_t* mail, hipStream_t s);
void launch_expand(const void* in, const int32_t* children, int64_t n_children,
                   const int32_t* oct_start, int32_t n_seg, const float* smin, const float* srg,
                   float mn1, float rg1, OctNode* out, hipStream_t s);

}  // namespace ocp
