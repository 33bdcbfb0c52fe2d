// Host-side launch wrappers for the gfx950 kernels.  Each takes plain device
// pointers and the stream to launch on; none allocates or synchronises.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace nbg {

// Radix-sort geometry (onesweep): 256 threads x sort_items(n) keys per tile.
// Fewer keys a thread while more would leave the chip short of tiles: a pass
// over u64 keys takes 6.7 us with 4 keys a thread and 11.0 with 16 at 10,000
// keys, 16.8 with 8 and 18 with 16 at 500,000, 27 with 8 and 23 with 16 at
// 1,048,576.
constexpr int kSortBlock = 256;
constexpr int64_t kSortSmall = (int64_t)1 << 18, kSortMedium = (int64_t)1 << 19;
constexpr int sort_items(int64_t n) { return n <= kSortSmall ? 4 : n <= kSortMedium ? 8 : 16; }
constexpr int kRadix = 256;

constexpr int64_t sort_tiles(int64_t n) {
    const int64_t tile = (int64_t)kSortBlock * sort_items(n);
    return (n + tile - 1) / tile;
}
// The most tiles of any n' <= n (a smaller sort may use smaller tiles).
constexpr int64_t sort_tiles_upto(int64_t n) {
    int64_t t = sort_tiles(n);
    if (n > kSortSmall && sort_tiles(kSortSmall) > t) t = sort_tiles(kSortSmall);
    if (n > kSortMedium && sort_tiles(kSortMedium) > t) t = sort_tiles(kSortMedium);
    return t;
}
constexpr int sort_passes(int key_bits) { return (key_bits + 7) / 8; }
// Words of status memory one sort needs: histograms, tile counters, the list
// of long runs, what the sort of all keys after a long run counts in, and per
// pass the tiles' look-back words (that sort uses three passes' of them, for
// tiles that are no smaller).
constexpr int kSortLongRuns = 4096, kSortAllPasses = 13;
constexpr int64_t kSortHeadWords = 8 * kRadix + 64 + 2 * kSortLongRuns + (kSortAllPasses + 1) * kRadix;
constexpr int64_t sort_status_words(int64_t n, int key_bits) {
    return kSortHeadWords + (int64_t)sort_passes(key_bits) * (sort_tiles_upto(n) * kRadix);
}

// How n keys of `bits` significant bits are sorted: `passes` radix passes over
// the bits from `shift` up, from the _alt buffers if from_alt, then (runs) the
// runs of keys that share those bits put in order.  Results land in the
// primary buffers.  lo: the keys have a low word too.
struct SortPlan {
    int passes, shift;
    bool runs, from_alt;
};
inline SortPlan sort_plan(int64_t n, int bits, bool lo) {
    const int full = sort_passes(bits);
    int need = 10;  // log2 n + 10 bits tell most bodies' spatial keys apart
    while (((int64_t)1 << (need - 10)) < n) ++need;
    SortPlan p;
    p.passes = sort_passes(need) < full ? sort_passes(need) : full;
    // A last pass costs what ranking the runs does, and no run can be long
    // (73,000 bodies of a forest, 34-bit keys: cells of the cores hold
    // hundreds, and sorting those runs took 2 ms, a pass takes 12 us).
    if (p.passes + 1 == full && !lo) p.passes = full;
    p.shift = bits > 8 * p.passes ? bits - 8 * p.passes : 0;
    p.runs = p.shift > 0 || lo;
    // the last kernel reads the _alt buffers (runs), or the last pass writes the primary ones
    p.from_alt = p.runs ? (p.passes & 1) == 0 : (p.passes & 1) != 0;
    return p;
}
// Words of status memory that a planned sort of n keys uses (to be cleared first).
inline int64_t sort_clear_words(int64_t n, const SortPlan &p) {
    return kSortHeadWords + (int64_t)p.passes * sort_tiles(n) * kRadix;
}

// Scan geometry.
constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanBlock * kScanItems;

// Ranges of words that a build sets before its first use of them, in one
// launch instead of one each.
struct FillRanges {  // what a kernel takes
    struct Range {
        uint32_t *p;
        int64_t n;
        uint32_t v;
    };
    Range r[10];
    int k = 0;
};
struct FillSet : FillRanges {
    std::vector<Range> more;  // ranges past the kernel's ten: a launch each
    void add(void *p, int64_t n, uint32_t v = 0u) {
        if (n <= 0) return;
        const Range q{(uint32_t *)p, n, v};
        if (k < 10) r[k++] = q;
        else more.push_back(q);
    }
};
void launch_fills(const FillSet &f, hipStream_t s);

// Body count above which the tree arrays' 32-bit indices would overflow.
constexpr int64_t kMaxBodies = (int64_t)1 << 29;




// One tree node as the walk reads it (48 bytes; the two children of a node
// are adjacent, so a sibling pair is 96 contiguous bytes):
//   mac  = LBVH: bbox centre xyz, squared bbox diagonal;
//   com  = centre of mass xyz, total mass;
//   topo = first body (sort order), body count, first child (-1 for a
//          leaf; the second child is first child + 1), parent (-1 root).
struct NodeRec {
    float4 mac;
    float4 com;
    int4 topo;
};

// One octree node as the walk reads it (64 bytes).  The non-empty children
// of a node are contiguous, in the reference's child order (octant
// 4x + 2y + z; empty octants have no record):
//   com  = centre of mass xyz, total mass;
//   lo   = cell centre - side (xyz), w = squared-distance opening threshold;
//   hi   = cell centre + side (xyz), w = bits of (octant | nchild << 8 |
//          level << 16);
//   topo = first body, body count, first child (-1 for a leaf), parent.
struct OctRec {
    float4 com;
    float4 lo;
    float4 hi;
    int4 topo;
};

__host__ __device__ inline int oct_nchild(const OctRec &r) { return (int)((__builtin_bit_cast(uint32_t, r.hi.w) >> 8) & 0xFFu); }
__host__ __device__ inline int oct_octant(const OctRec &r) { return (int)(__builtin_bit_cast(uint32_t, r.hi.w) & 0xFFu); }
__host__ __device__ inline int oct_level(const OctRec &r) { return (int)(__builtin_bit_cast(uint32_t, r.hi.w) >> 16); }

// Octree key geometry: the octant of every level is a 3-bit digit; levels
// 0..20 live in key_hi bits 62..0, levels 21..33 in key_lo bits 38..0.
constexpr int kOctHiLevels = 21;
constexpr int kOctLevels = 34;   // max_depth 32 below the two forced levels
constexpr int kOctThrStride = 64;  // opening thresholds per system (one per level)

// Upper bound on the number of non-empty octree nodes: every body is in one
// leaf, and on each level 2..levels-1 an internal node holds > leaf bodies.
inline int64_t octree_capacity(int64_t n, int leaf, int max_depth) {
    const int64_t levels = (int64_t)max_depth + 2;
    return 9 + n + (levels - 2) * (n / ((int64_t)leaf + 1) + 1);
}

// Work buffers of the octree build (capacity `cap` nodes, n bodies).
struct OctBuffers {
    int64_t cap = 0, n = 0;
    float4 *targets = nullptr;  // forests: the walk's targets in their order
    uint64_t *key_hi = nullptr, *key_lo = nullptr, *lo_sorted = nullptr;  // n each
    uint32_t *nown = nullptr;      // n: nodes whose range starts at a position
    uint32_t *nbase = nullptr;     // n: exclusive scan of nown (pre-order node ids)
    int32_t *nfirst = nullptr, *ncount = nullptr, *nparent = nullptr;  // cap, by node id
    uint32_t *nmeta = nullptr;     // cap: level | octant << 8 | leaf << 12
    uint32_t *occ = nullptr;       // cap: occupied-child octant mask
    uint32_t *cb = nullptr;        // cap: child counts, then their exclusive scan
    uint32_t *flags = nullptr;     // cap: summary arrival counters
    uint32_t *glist = nullptr;     // 2 * oct_queue_words(n): two queues of straddling parents (summaries)
    uint32_t *scan_ws = nullptr;   // the scan tiles' sums of nown, then of cb (oct_scan_words)
    OctRec *nodes = nullptr;       // cap, by slot
    float4 *centre = nullptr;      // cap, by slot: cell centre xyz, side
    float *thr = nullptr;          // 64: opening threshold per level
    uint32_t *misc = nullptr;      // 64: [0] node total, [1] child total
    uint32_t *sums_own() const { return scan_ws; }
    uint32_t *sums_child() const { return scan_ws + (n + kScanTile - 1) / kScanTile; }
};
// The summaries' queue: a place for each body, a count for each kOctSegment of them.
constexpr int kOctSegment = 1024;
inline int64_t oct_queue_words(int64_t n) { return n + (n + kOctSegment - 1) / kOctSegment; }
inline int64_t oct_scan_words(int64_t n, int64_t cap) {
    return (n + kScanTile - 1) / kScanTile + (cap + kScanTile - 1) / kScanTile + 1;
}
// What an octree build of n bodies counts in, to be set before it.
inline void oct_fills(FillSet &f, const OctBuffers &ob, int64_t n, int32_t *leaf_start) {
    f.add(ob.scan_ws, oct_scan_words(ob.n, ob.cap));
    f.add(ob.occ, ob.cap);
    f.add(leaf_start, n, 0xFFFFFFFFu);
    f.add(ob.flags, ob.cap);
}
// What a linear-BVH build of n bodies counts in, to be set before it.
inline void lbvh_fills(FillSet &f, int64_t n, int32_t *leaf_start, uint32_t *scan_ws, uint32_t *flags) {
    f.add(scan_ws, 64 + (n + kScanTile - 1) / kScanTile);
    f.add(leaf_start, n, 0xFFFFFFFFu);
    f.add(flags, 2 * n);
}

// Octree build (Octree::build, Trees/Octree.h:185-205) in three stages, each
// enqueue-only, after launch_bbox with oct_fills and the sort's words.
// keys: per-body octant path on the reference's float centre recurrence (the
// high word to the buffers that `plan` starts from, the low word to
// ob.key_lo) and the levels' opening thresholds.  sort: launch_sort with
// ob.key_lo / ob.lo_sorted when there is a low word.  topology: cells from
// the sorted keys, node records, leaf contents reordered by original index
// into idx (the final body order; idx_in is the key order), leaf_start.
// Summaries run after the body gather.
inline bool oct_has_lo(int max_depth) { return max_depth + 2 > kOctHiLevels; }
void launch_octree_keys(const float *x, const float *y, const float *z, int64_t n, const float *partials, int blocks,
                        float *bbox6, int max_depth, float theta, const SortPlan &plan, OctBuffers &ob, uint64_t *keys,
                        uint32_t *idx, uint64_t *keys_alt, uint32_t *idx_alt, uint32_t *status, hipStream_t s);
void launch_octree_topology(int64_t n, const float *bbox6, int leaf_size, int max_depth, OctBuffers &ob,
                            const uint64_t *keys, const uint32_t *idx_in, uint32_t *idx, int32_t *leaf_start,
                            uint32_t *err, hipStream_t s);
// Forest of octrees: bodies of system s (bsys, original order) get paths
// over their own system's cube (bbox6 + 6 s) and depth (lv_tab[s] levels);
// the sort orders positions by system, then path.  Leaves the sorted high
// words in keys (low words in ob.lo_sorted when max_levels > 21), the
// sorted system index in keys_alt and the permutation in idx_alt.
void launch_octree_forest_build(const float *x, const float *y, const float *z, int64_t n, int nsys,
                                const uint32_t *bsys, const float *bbox6, const int32_t *lv_tab, int max_levels,
                                OctBuffers &ob, uint64_t *keys, uint32_t *idx, uint64_t *keys_alt, uint32_t *idx_alt,
                                uint32_t *sort_status, uint32_t *err, hipStream_t s);

// Forest topology: every system gets its own octree (root slot s, its own
// leaf size, depth, and opening thresholds from its cube and theta =
// sys_prm[s].z; ob.thr holds kOctThrStride floats per system).
void launch_octree_forest_topology(int64_t n, int nsys, const float *bbox6, const float4 *sys_prm,
                                   const int32_t *lv_tab, const int32_t *leaf_tab, const int64_t *sys_first,
                                   int max_levels, OctBuffers &ob, const uint64_t *keys, const uint64_t *sys_sorted,
                                   const uint32_t *idx_alt, uint32_t *idx, int32_t *leaf_start, uint32_t *err,
                                   hipStream_t s);

// Per-system bounding boxes; part: scratch of 24 bytes for every 2,048 bodies
// (used if the largest system has more than 8,192).
void launch_seg_bbox(const float *x, const float *y, const float *z, int64_t n, int nsys, const int64_t *sys_first,
                     int64_t largest, float *bbox6, float *part, hipStream_t s);

void launch_octree_summaries(const float4 *bodies, int64_t n, OctBuffers &ob, const int32_t *leaf_start,
                             uint32_t *err, hipStream_t s, float4 *quad = nullptr);

void launch_fill_u32(uint32_t *p, uint32_t v, int64_t n, hipStream_t s);

// Exclusive scan of n > 0 u32 values into out (in may equal out) from the
// tiles' sums (ceil(n / kScanTile) words, overwritten); total receives the
// sum.  nlim (or null): a device count of items, those past it being zero.
// Up to kScanFused items the kernel that computes them adds up the tiles'
// sums (one launch less; measured: 4 us less at 10,000 items, 20 us more at
// 1,048,576, where the waves' atomics meet).
constexpr int kScanFold = 4096;
constexpr int64_t kScanFused = (int64_t)1 << 18;
inline bool scan_fused(int64_t n) { return n <= kScanFused; }
void launch_scan_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *sums, uint32_t *total, hipStream_t s,
                     const uint32_t *nlim = nullptr);

// Stable radix sort of u64 keys + u32 payload over the low 8 * passes bits.
// Returns true when the result is in the _alt buffers (odd passes).
bool launch_radix_sort_u64(uint64_t *keys, uint32_t *idx, uint64_t *keys_alt, uint32_t *idx_alt, int64_t n,
                           int passes, uint32_t *status, uint32_t *err, hipStream_t s);

// outerBoundingBox, first stage: per-block partials (6 * kBBoxBlocks floats),
// and the ranges in `fills` set.  Returns the number of partials; the kernel
// that computes the keys folds them and stores the box.
constexpr int kBBoxBlocks = 512;
int launch_bbox(const float *x, const float *y, const float *z, int64_t n, float *partials, const FillSet &fills,
                hipStream_t s);

// Morton keys (bits = 30 -> u32 keys, 63 -> u64 keys) and iota payload into
// the buffers that `plan` starts from, with the sort's histograms in `status`
// (cleared).  blocks > 0: the box is folded from that many partials and
// stored in bbox6; 0: bbox6 holds it.
void launch_morton(const float *x, const float *y, const float *z, int64_t n, const float *partials, int blocks,
                   float *bbox6, int bits, const SortPlan &plan, void *keys, uint32_t *idx, void *keys_alt,
                   uint32_t *idx_alt, uint32_t *status, hipStream_t s);

// Stable sort of (key, idx) as planned (keys in place, status cleared and
// with the histograms).  The result is in keys / idx.  lo (u64 keys): the
// keys' low words by original index, lo_sorted receives them in key order.
// err is a device flag word.
void launch_sort(void *keys, uint32_t *idx, void *keys_alt, uint32_t *idx_alt, int64_t n, int bits,
                 const SortPlan &plan, uint32_t *status, uint32_t *err, hipStream_t s, const uint64_t *lo = nullptr,
                 uint64_t *lo_sorted = nullptr);

// Sorted SoA -> float4 (x, y, z, m) in sort order.
void launch_gather(const float *x, const float *y, const float *z, const float *m, const uint32_t *perm,
                   int64_t n, float4 *bodies, hipStream_t s);

// LBVH topology (Karras radix tree truncated at the reference's leaf rule)
// into the compact node arrays, and the bodies in key order (perm).  scratch
// ints: first, last, gamma, split, rank, parent (6 * n words) plus scan_ws
// (64 words and the scan tiles' sums, cleared); leaf_start is set to -1
// before.  node_count receives the number of nodes.
void launch_lbvh_topology(const void *keys, int bits, int64_t n, int leaf_size, int32_t *kfirst,
                          int32_t *klast, int32_t *kgamma, uint32_t *ksplit, uint32_t *krank,
                          int32_t *kparent, uint32_t *scan_ws, NodeRec *nodes, int32_t *leaf_start,
                          uint32_t *node_count, const float *x, const float *y, const float *z, const float *m,
                          const uint32_t *perm, float4 *bodies, hipStream_t s, int sys_shift = 0,
                          const int32_t *leaf_tab = nullptr);

// Bottom-up LBVH summaries with atomic arrival flags: COM, mass, bbox and the
// MAC record (bbox centre, squared diagonal).  leaf_start[i] holds the leaf
// slot whose first body is i (else -1; written by the topology pass);
// flags holds max_nodes words; glist holds 2 * (2n + 64) words (two queues
// and their counts).
constexpr int kSummBodies = 512;   // bodies per workgroup in the local pass, one per thread
struct MacParam {       // mac_threshold's output for one theta
    double mid;
    int tie;
};
// mp_tab (forest): per-system MAC parameters, indexed by keys[first] >> sys_shift.
// quad (quadrupole trees): 2 * max_nodes float4 of second moments (layout in
// device.hpp), or null.
void launch_lbvh_summaries(const float4 *bodies, int64_t n, NodeRec *nodes, const int32_t *leaf_start,
                           int64_t max_nodes, uint32_t *flags, uint32_t *glist, float4 *bmin, float4 *bmax,
                           float theta, uint32_t *err, hipStream_t s, const MacParam *mp_tab = nullptr,
                           const uint64_t *keys = nullptr, int sys_shift = 0, float4 *quad = nullptr);

// Forest of independent systems (30-bit codes, u64 keys = system << 30 | code):
// per-system bounding boxes (bbox6: 6 floats per system), keys, and one sort;
// sets `fills` and the sort's words first.
void launch_forest_build(const float *x, const float *y, const float *z, int64_t n, int nsys,
                         const int64_t *sys_first, int64_t largest, const uint32_t *bsys, float *bbox6, uint64_t *keys, uint32_t *idx,
                         uint64_t *keys_alt, uint32_t *idx_alt, uint32_t *sort_status, FillSet &fills, uint32_t *err,
                         hipStream_t s);
// sys_root[s] = slot of the node whose range is exactly system s.
void launch_forest_roots(const NodeRec *nodes, const uint32_t *node_count, int64_t max_nodes, const uint64_t *keys,
                         int64_t n, int nsys, int32_t *sys_root, uint32_t *err, hipStream_t s);
// Forest update: dt of body i is sys_prm[bsys[i]].w.
void launch_update_forest(float *x, float *y, float *z, float *vx, float *vy, float *vz, const float *ax,
                          const float *ay, const float *az, const uint32_t *bsys, const float4 *sys_prm, int64_t n,
                          hipStream_t s);

// Forest non-finite guard: bad[bsys[i]] = 1 for every body i whose position
// or velocity is NaN or infinite (bad is cleared by the caller).
void launch_forest_nonfinite(const float *x, const float *y, const float *z, const float *vx, const float *vy,
                             const float *vz, const uint32_t *bsys, int64_t n, uint32_t *bad, hipStream_t s);

// Host side of mac_lbvh_exact: the FP64 midpoint below T = RN(theta*theta)
// and whether a tie rounds down (T has an odd significand).
inline void mac_threshold(float theta, double *mid, int *tie) {
    const float T = theta * theta;
    if (!(T > 0.0f)) { *mid = -1.0; *tie = 0; return; }
    uint32_t bits;
    __builtin_memcpy(&bits, &T, 4);
    const uint32_t pbits = bits - 1;  // predecessor of a positive finite float
    float P;
    __builtin_memcpy(&P, &pbits, 4);
    *mid = ((double)P + (double)T) * 0.5;
    *tie = (int)(bits & 1u);
}

struct WalkArgs {
    int64_t n;              // bodies in the tree
    const float4 *bodies;   // sorted (x, y, z, m)
    int64_t nt;             // targets walked (the bodies themselves, or passive points)
    const float4 *targets;  // targets in walk order (xyz)
    const uint32_t *perm;   // walk position -> output index (< nt)
    const NodeRec *nodes;   // LBVH nodes
    const OctRec *onodes;   // octree nodes
    int levels;             // octree: max_depth + 2
    float theta;            // octree MAC
    float theta2;           // LBVH MAC: theta * theta (float)
    double mac_mid;         // LBVH MAC threshold (mac_threshold)
    int mac_tie;
    float G, eps2;
    int64_t max_nodes;      // node array capacity (index guard)
    float *ax, *ay, *az;    // output order (nt each)
    unsigned long long *counts;  // [pp, np]
    uint32_t *err;
    // Forest walk (nsys > 0): waves are aligned to systems.  Wave w serves
    // system s with wave_first[s] <= w < wave_first[s+1], targets
    // sys_first[s] + 64 (w - wave_first[s]) + lane below sys_first[s+1],
    // starts at node sys_root[s] and uses G = sys_prm[s].x, eps2 = sys_prm[s].y.
    int nsys = 0;
    int64_t nwaves = 0;
    const int64_t *wave_first = nullptr;
    const int64_t *sys_first = nullptr;
    const int32_t *sys_root = nullptr;
    const float4 *sys_prm = nullptr;
    // Quadrupole trees: second moments per node slot (2 float4, layout in
    // device.hpp); null for monopole trees.
    const float4 *quad = nullptr;
    // Waves that share 16 targets.  FAST: 1, 2 or 4.  ORDERED: 8 or 16 by
    // frames (2 and 4 read as 8), 1: the recursion, 64 targets a wave.
    // ORDERED with split_part_f: that many waves per 64 targets, which leave
    // their frontier subtrees' results there (kOrderedSplitSlots x 3 floats
    // per target, split_stride floats apart) for a second kernel.
    int split = 1;
    float *split_part_f = nullptr;
    int64_t split_stride = 0;
};

// Walks of systems from this size on take their targets in compact groups
// (targets.hip).  Below, the pass that forms them costs what it saves; walk
// and pass, us, without / with: octree 80,000 bodies 246 / 278, 131,000 340 /
// 360, 160,000 409 / 387; linear BVH 64,000 438 / 442, 131,000 794 / 784.
constexpr int64_t kGroupMin = 160000;
// The ORDERED recursion, one wave per 64 targets, gains later, when its waves
// no longer end together; walk ms, without / with: octree 300,000 bodies 6.6 /
// 7.4, 400,000 7.4 / 7.6, 600,000 10.9 / 10.8, 1,000,000 15.9 / 14.9; linear BVH
// 200,000 9.9 / 10.2, 400,000 15.0 / 14.5, 600,000 20.9 / 20.2.  (By frames,
// octree 200,000 4.9 / 4.6.)
constexpr int64_t kGroupMinChains = 500000;
void launch_group_targets(const float4 *bodies, const uint32_t *perm, int64_t n, float4 *out, uint32_t *out_perm,
                          hipStream_t s);
// A forest's: systems below kGroupMin keep their order.
void launch_group_targets_forest(const float4 *bodies, const uint32_t *perm, int64_t n, const int64_t *sys_first,
                                 int nsys, float4 *out, uint32_t *out_perm, hipStream_t s);

// Rows of floats that are copied to or from the host together; xyz: the last
// three go out interleaved.
struct RowSet {
    float *row[10] = {};
    int k = 0;
    bool xyz = false;
};
// Elements i0 .. i0 + cnt - 1 of every row to words 0 .. k * stride - 1 (pinned
// host memory, row j from j * stride on; stride a multiple of 4), and *err
// (may be null) to *err_out.
void launch_rows_out(const RowSet &R, int64_t i0, int cnt, int stride, float *words, const uint32_t *err,
                     uint32_t *err_out, hipStream_t s);
// The other way; rows in `absent` are cleared.
void launch_rows_in(const RowSet &R, int cnt, int stride, const float *words, uint32_t absent, hipStream_t s);

// ORDERED waves per 16 targets for a walk by frames of `groups` groups of 64
// targets, 1: none.  Measured, walk us at n bodies, theta 0.5, leaf 16:
// octree, 8 / 16 waves / recursion (the split that was here before): 1,000 59
// / 49 / 315; 3,000 94 / 102; 10,000 235 / 294 / 1,045; 200,000 3,777 / 5,685
// / 5,393; 400,000 8,911 / - / 7,426.  Linear BVH, 8 / 16 / split: 3,000 142 /
// 118 / 478; 5,000 272 / 267 / 720; 10,000 891 / 987 / 1,026; 16,000 1,457 /
// 2,407 / 1,595: its frames outgrow the slots.
// The recursion's time is the chain of its largest tree, `bodies`, which a
// forest's other groups hide behind; the frames' grows with the groups.  A
// step of octrees of 64 / 1,000 / 3,000 / 11,000 bodies, ms, recursion : 8
// waves, at 128 groups 0.34 : 0.37, 0.90 : 0.43, 1.66 : 0.45, -; 512 0.38 :
// 0.66, 0.94 : 0.79, 1.69 : 0.83, 3.1 : 0.9; 1,024 0.43 : 1.05, 0.97 : 1.24, 1.75
// : 1.34, 3.2 : 1.3; 4,096 0.66 : 3.3, 1.4 : 3.8, 2.4 : 4.2, 4.3 : 4.1.  Linear
// BVHs of 64 bodies, 128 and 256 groups 0.130 : 0.125 and 0.135 : 0.155.
inline int64_t ordered_frames_most(bool octree) { return octree ? 4096 : 256; }
inline int ordered_split_waves(int64_t groups, bool octree, int64_t bodies) {
    if (groups > ordered_frames_most(octree) || groups > 64 + bodies / 2) return 1;
    return groups <= (octree ? 32 : 80) ? 16 : 8;
}

// ORDERED split of one linear BVH of n bodies past that: waves per 64 targets
// within 4,096 waves (1: the chip is full without), one result per frontier
// subtree.
constexpr int kOrderedSplitSlots = 128;
constexpr int64_t kOrderedSplitMaxBodies = 65536;
inline int ordered_subtree_waves(int64_t n) {
    const int64_t groups = (n + 63) / 64;
    if (ordered_split_waves(groups, false, n) > 1 || n > kOrderedSplitMaxBodies) return 1;
    int k = 1;
    while (k < 16 && groups * 2 * k <= 4096) k *= 2;
    return k;
}
// FAST waves per 16 targets for a walk of `groups` groups of 64 targets: the
// most, up to 4, that keep the launch within 4,096 waves (4 per SIMD).
inline int fast_split_waves(int64_t groups) {
    int k = 1;
    while (k < 4 && groups * 4 * k * 2 <= 4096) k *= 2;
    return k;
}

// Barnes-Hut traversal over the LBVH.  ordered != 0 selects the
// bit-exact reference arithmetic; diag != 0 makes the FAST walk also count
// its schedule statistics (counts[2..5]).
void launch_walk_lbvh(const WalkArgs &a, int ordered, int max_depth, int diag, hipStream_t s);

// Barnes-Hut traversal over the octree (same modes and statistics).
void launch_walk_oct(const WalkArgs &a, int ordered, int diag, hipStream_t s);

// The FAST walks of both trees (walk_fast.hip).
void launch_walk_fast(const WalkArgs &a, bool octree, int stats, hipStream_t s);

// Implicit FMM (fmm.hip): the lockstep dual traversal breadth-first, one
// launch per traversal step, then one launch for the passive leaves.
// Frontier items (kFmmItemWords each) alternate between two halves by step
// parity; ctr holds three rotating sets of {items, next item, -, -}; leaf
// groups collect in `groups` for the last launch; lists live in one pool for
// the whole pass.  counts: [pp, np, pn, nn]; err bit 16: a list, the frontier
// or the leaf groups outgrew their capacity.
constexpr int kFmmItemWords = 16;
constexpr int kFmmGroupWaves = 8192;  // the leaf-group launch (8 waves per SIMD)
constexpr int kFmmUlistCap = 4096;    // close active nodes kept per leaf-group wave
constexpr int kFmmStartCap = 512;
constexpr int kFmmSeedWaves = 272;  // one per starting node (at most 256 + 7)
struct FmmArgs {
    int64_t n;
    const float4 *bodies;     // tree order (x, y, z, m)
    const OctRec *nodes;
    const float4 *centre;     // cell centre xyz, side, by slot
    const uint32_t *misc;     // octree misc ([0] node count)
    int64_t max_nodes;
    const uint32_t *perm;     // tree position -> original index
    float *ax, *ay, *az;
    float theta, G, eps2;
    // the criteria's bounds on FP32 quotients (fmm.hip's quotient_below): the
    // midpoints below theta * theta and below theta (set by launch_fmm)
    double theta2_mid, theta_mid;
    int32_t *starts;          // kFmmStartCap
    uint32_t *nstarts;
    uint32_t *ctr;            // 12 words
    uint32_t *pool_ctr;       // pool words used
    uint32_t *group_ctr;      // [0] leaf groups, [1] next leaf group
    uint32_t *peak;           // 4 words: pool words, items (largest step), steps run
    uint32_t *items[2];       // item_cap items each
    uint32_t *groups;         // item_cap items
    uint32_t *pool;           // pool_cap words
    int64_t item_cap, pool_cap;
    uint32_t *seed_scratch;   // kFmmSeedWaves x 3 x cap_a words
    uint32_t *ulist;          // kFmmGroupWaves x ulist_cap node slots
    int ulist_cap;
    int cap_a, waves, steps;
    unsigned long long *counts;
    uint32_t *err;
};
void launch_fmm(const FmmArgs &a, hipStream_t s);

// v = v + a*dt; p = p + v*dt (original order).
void launch_update(float *x, float *y, float *z, float *vx, float *vy, float *vz, const float *ax,
                   const float *ay, const float *az, float dt, int64_t n, hipStream_t s);

// NaiveSolver in FP32: every target sums every source in order (ORDERED:
// the reference's exact arithmetic).  Result of target i goes to
// out_index[i] (or i when out_index is null).
void launch_direct_f32(const float4 *src, int64_t ns, const float4 *tgt, int64_t nt, const uint32_t *out_index,
                       float G, float eps2, int ordered, float *ax, float *ay, float *az, hipStream_t s);

// FP64 direct sum at targets (float4 sources x,y,z,m; targets float4 x,y,z).
void launch_direct_f64(const float4 *src, int64_t ns, const float4 *tgt, int64_t nt, double G, double eps2,
                       double *ax, double *ay, double *az, hipStream_t s);

// SoA (x, y, z, m) -> float4, original order.
void launch_pack(const float *x, const float *y, const float *z, const float *m, int64_t n, float4 *out,
                 hipStream_t s);

// FP64 softened potential, each pair i < j once: wave w (64 targets) of
// [w0, w1) writes sum_{i in wave} m_i sum_{j > i} m_j / sqrt(r^2 + eps2)
// into partial[w]; -G times the sum of all potential_waves(n) partials is
// the potential.  bodies: (x, y, z, m) in FP64 (launch_pack_f64).
int64_t potential_waves(int64_t n);
void launch_pack_f64(const float *x, const float *y, const float *z, const float *m, int64_t n, double4 *out,
                     hipStream_t s);
void launch_potential_f64(const double4 *bodies, int64_t n, double eps2, int64_t w0, int64_t w1, double *partial,
                          hipStream_t s);

}  // namespace nbg
