// Barnes-Hut traversal for gfx950.
//
// One wavefront walks the tree for 64 spatially adjacent targets (consecutive
// in Morton order).  At every node, each lane in the wave's active mask
// evaluates its own opening criterion; lanes that accept the node take its
// monopole, lanes that reject a leaf interact with its bodies, and lanes that
// reject an internal node (a ballot) form the mask with which its children
// are visited.  Each lane therefore meets exactly the nodes and bodies the
// reference's per-body recursion meets (Descent/activeTree.h:24-79); only the
// schedule is shared.  Node records and leaf bodies are wave-uniform and are
// read with scalar loads.
//
// ORDERED (bit-exact): depth-first in child order with completion markers on
// an LDS stack, IEEE sqrt/division in Gravity::particleParticle's order
// (Physics/Rules/Gravity.h:199-209), leaf sums sequential from zero
// (activeTree.h:44-52) and child results bracketed as libstdc++'s
// std::transform_reduce does for two children, (0 + r0) + r1
// (activeTree.h:66-76).  Each lane's pending partial sums of the open depths
// (the depth is wave-uniform) sit in an LDS ring for the deepest levels and a
// private array for the rest (linear BVH), or in registers for the top frame
// and a private array below it (octree).  A subtree's result does not depend
// on where it is computed, so the walks of small systems compute it where
// there is room, with unchanged bits: by frames, or frontier subtrees walked
// from zero by several waves.
//
// The FAST walks (walk_fast.hip) take the same opening decisions in another
// schedule.

#include "device.hpp"
#include "launch.hpp"
#include "walk_common.hpp"
#include "walk_task.hpp"

#include <type_traits>

namespace nbg {

constexpr int kMetaComplete = 0x10000;
// Upper bound on loop iterations per wave; a valid tree needs at most ~3 per node.
constexpr uint32_t kMaxWalkIters = 1u << 28;

// DiagonalOverCenterDistance (DiagonalOverCenterDistance.h:18-22) for one
// lane: the squared distance to the bbox centre in glm's order, compared
// with the node's threshold (mac_lbvh_threshold, computed with the node's
// summary), which is exactly equivalent to diag2 / d2 < theta^2 in FP32.
__device__ __forceinline__ bool lbvh_accepts(float4 mc, float px, float py, float pz) {
    const float dx = px - mc.x, dy = py - mc.y, dz = pz - mc.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    return d2 > mc.w;
}

// ---------------------------------------------------------------- ORDERED
constexpr int kOrderedWaves = 4;  // waves per workgroup of the ORDERED walks

// Two ways to lay out an ORDERED wave.  64 targets: lane = target.  ROWS: 16
// targets, each in the same lane of the four 16-lane rows; a leaf's bodies are
// evaluated four at a time, one per row, and added in order.  The walks by
// frames are in ROWS: four times the waves for a small system, and a quarter
// of the serial chain of a leaf's evaluations.
constexpr int kRowTargets = 16;
template <bool ROWS>
__device__ __forceinline__ int target_bit() { return ROWS ? lane_id() & (kRowTargets - 1) : lane_id(); }
template <bool ROWS>
__device__ __forceinline__ uint64_t target_ballot(bool p) {
    const uint64_t b = __ballot(p);
    return ROWS ? b & 0xFFFFull : b;
}

// v of each row, in every row (same lane of the row).
__device__ __forceinline__ void spread_rows(float v, float (&o)[4]) {
    const uint32_t u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);  // rows 0 0 2 2 and 1 1 3 3
    const auto e = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
    const auto d = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
    o[0] = __uint_as_float(e[0]);
    o[1] = __uint_as_float(d[0]);
    o[2] = __uint_as_float(e[1]);
    o[3] = __uint_as_float(d[1]);
}

// A leaf's sum, sequential from zero over its bodies (activeTree.h:44-52),
// for the lanes with `op` (ROWS: in every row).
template <bool ROWS>
__device__ __forceinline__ void leaf_ordered(const float4 *__restrict__ bodies, int first, int cnt, bool op, float px,
                                             float py, float pz, float G, float eps2, float &lx, float &ly, float &lz) {
    lx = 0.0f; ly = 0.0f; lz = 0.0f;
    if constexpr (ROWS) {
        const int row = lane_id() / kRowTargets;
        // W bodies of every row in flight
        auto block = [&](auto width, int j) {
            constexpr int W = decltype(width)::value;
            float vx[W], vy[W], vz[W];
#pragma unroll
            for (int h = 0; h < W; ++h) {
                const int i = j + 4 * h + row;
                const float4 b = bodies[first + (i < cnt ? i : cnt - 1)];
                pp_exact(b.x, b.y, b.z, b.w, px, py, pz, G, eps2, vx[h], vy[h], vz[h]);
            }
#pragma unroll
            for (int h = 0; h < W; ++h) {
                if (j + 4 * h >= cnt) break;
                float x[4], y[4], z[4];
                spread_rows(vx[h], x);
                spread_rows(vy[h], y);
                spread_rows(vz[h], z);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (j + 4 * h + q >= cnt) break;
                    lx = lx + x[q]; ly = ly + y[q]; lz = lz + z[q];
                }
            }
        };
        int j = 0;
        for (; cnt - j > 8; j += 16) block(std::integral_constant<int, 4>{}, j);
        for (; cnt - j > 4; j += 8) block(std::integral_constant<int, 2>{}, j);
        if (cnt > j) block(std::integral_constant<int, 1>{}, j);
    } else {
        // the body loop runs in wave-uniform flow so its loads are scalar
        // (one per body for the wave); the opened lanes sum
        for (int j = 0; j < cnt; ++j) {
            const float4 b = bodies[first + j];
            if (op) {
                float vx, vy, vz;
                pp_exact(b.x, b.y, b.z, b.w, px, py, pz, G, eps2, vx, vy, vz);
                lx = lx + vx; ly = ly + vy; lz = lz + vz;
            }
        }
    }
}

// ---- ORDERED by frames (small systems): a workgroup of K waves per 16
// targets.  A frame is a node that some of the 16 targets open; its result
// needs those of its children only.  First the frames are listed, a level of
// the tree at a time, by the opening criterion alone; then they are evaluated
// from the last level up, each by one wave (accepted children side by side in
// the rows, opened leaves by leaf_ordered, opened nodes' results from LDS) and
// bracketed as the recursion does.  A frame's result does not depend on when
// or where it is computed.  What the slots have no room for is walked by the
// recursion: the linear BVH stops listing before a level whose children might
// not fit and its waves take that level's frames in turn; an octree frame's
// children past the last slot are walked in the frame's evaluation.
//
// Against the recursion, which meets its nodes one after the other, each with
// the latency of a record's load, a square root and a division (10,000
// bodies, octree, theta 0.5, leaf 16: some 1,400 steps per 64 targets), a
// level's frames are independent of one another and the waves share them
// whatever the tree's shape.  Measured against the recursion split by
// subtrees: 10,000 bodies, octree, 1,045 -> 235 us; 1,000 bodies, linear BVH,
// theta 0.3, leaf 64, 169 -> 52 us.  Bound by the levels' latency at 1,000,
// then by vector issue and the waits at each level's end.
template <int kSlots>
struct Frames {
    float part[kSlots][3][kRowTargets];  // results: the frames', then the listed leaves'
    int child[kSlots];                   // a frame's first child; a leaf
    uint16_t mask[kSlots];               // targets that open it
    uint16_t kids[kSlots];               // children that are frames (low 8 bits), number of children (above)
    uint16_t slot[kSlots];               // their first frame
    uint8_t items[kSlots];               // children that are listed leaves
    uint16_t islot[kSlots];              // their first listed leaf
    int first[66];                       // the levels' first frames
    int tail, itail, next;
};
// As many frames as the LDS of a CU has room for beside the waves' own bytes,
// with 2 workgroups of 8 waves or 1 of 16 on the CU (LDS is given out
// in units of 1,280 bytes).
constexpr int frames_of(int waves, int wave_bytes) {
    const int lds = waves >= 16 ? 128 * 1280 : 64 * 1280;
    return (lds - waves * wave_bytes - 512) / (3 * kRowTargets * 4 + 13);
}
// With 16 waves per 16 targets the chip is far from full and a level's time
// is its longest wave's: opened leaves are listed too, as items, and summed
// before the frames.  With fewer waves the slots all go to frames and a leaf
// is summed in its parent's evaluation.
constexpr int items_of(int waves, int slots) { return waves >= 16 ? slots * 2 / 5 : 0; }

// ---- ORDERED split: the top of a linear BVH is its internal nodes above
// depth kTopDepth that hold more than `cut` bodies; the top nodes' other
// children are the frontier, at most 2^kTopDepth nodes.
constexpr int kTopDepth = 7;
constexpr int kMaxFrontier = 1 << kTopDepth;
static_assert(kMaxFrontier == kOrderedSplitSlots, "ORDERED split: one slot per frontier entry");

__device__ __forceinline__ bool lbvh_top(const NodeRec &r, int depth, int cut) {
    return r.topo.z >= 0 && r.topo.y > cut && depth < kTopDepth;
}

constexpr int kSaveRing = 4;
constexpr int kRowsRing = 8;  // of the walk by frames
// lanes of a ring's level: in ROWS every row holds the same
template <bool ROWS>
constexpr int kRingLanes = ROWS ? kRowTargets : kWave;

// The ORDERED descent from node `start` for the lanes of `smask`, the
// reference's recursion (activeTree.h:24-79) with its bracketing: each node's
// result into r (from zero), counts into cpp / cnp.  RING: levels of the LDS
// ring.  TOP: a visited node that is not a top node (lbvh_top with the root's
// cut) is a frontier node: its result is not walked but taken from
// split_part_f (slot fi, counted in visit order) and added as the walk would
// add it.
template <int MAXD, bool QUAD, bool ROWS, int RING, bool TOP = false>
__device__ __forceinline__ void ordered_descent(const WalkArgs &a, int start, uint64_t smask, float px, float py,
                                                float pz, float G, float eps2, int *s_node, int *s_meta,
                                                uint64_t *s_mask, float *ring, float &rx, float &ry, float &rz,
                                                uint32_t &cpp, uint32_t &cnp, bool &fail,
                                                int64_t tgt = 0, int cut = 0) {
    constexpr int kStack = 2 * MAXD + 4;
    constexpr int kL = kRingLanes<ROWS>;
    float s_save[MAXD * 3];
    const float4 *__restrict__ bodies = a.bodies;
    const NodeRec *__restrict__ nodes = a.nodes;
    const int lane = lane_id(), bit = target_bit<ROWS>();
    int fi = 0;
    if (lane == 0) { s_node[0] = start; s_meta[0] = 0; s_mask[0] = smask; }
    __builtin_amdgcn_wave_barrier();
    int sp = 1;
    int ring_base = 0;
    uint32_t iters = 0;
    while (sp > 0) {
        if (++iters > kMaxWalkIters) { fail = true; break; }
        --sp;
        __builtin_amdgcn_wave_barrier();
        const int node = uniform_i32(s_node[sp]);
        const int meta = uniform_i32(s_meta[sp]);
        const uint64_t mask = uniform_u64(s_mask[sp]);
        const bool act = (mask >> bit) & 1ull;
        const int depth = meta & 0xFFFF;
        if (meta & kMetaComplete) {
            // the deepest pending depth comes back: from the ring, or (the
            // ring then holds nothing) from scratch
            if (depth >= ring_base) {
                const float *slot = ring + (depth % RING) * 3 * kL + bit;
                if (act) {
                    const float vx = rx, vy = ry, vz = rz;
                    rx = slot[0] + vx;
                    ry = slot[kL] + vy;
                    rz = slot[2 * kL] + vz;
                }
            } else {
                ring_base = depth;
                if (act) {
                    const float vx = rx, vy = ry, vz = rz;
                    rx = s_save[depth * 3 + 0] + vx;
                    ry = s_save[depth * 3 + 1] + vy;
                    rz = s_save[depth * 3 + 2] + vz;
                }
            }
            continue;
        }
        if (node < 0 || node >= a.max_nodes) { fail = true; break; }
        const NodeRec nd = nodes[node];
        if (TOP && !lbvh_top(nd, depth, cut)) {
            // a frontier node: its subtree's result, walked from zero elsewhere
            if (fi >= kMaxFrontier) { fail = true; break; }
            if (act) {
                const int64_t o = (int64_t)fi * 3 * a.split_stride + tgt;
                const float vx = a.split_part_f[o], vy = a.split_part_f[o + a.split_stride],
                            vz = a.split_part_f[o + 2 * a.split_stride];
                rx = rx + vx; ry = ry + vy; rz = rz + vz;
            }
            ++fi;
            continue;
        }
        const bool pass = act && lbvh_accepts(nd.mac, px, py, pz);
        if (pass) {
            ++cnp;
            float vx, vy, vz;
            if (QUAD)
                np_quad_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, a.quad[2 * node], a.quad[2 * node + 1], px, py,
                              pz, G, eps2, vx, vy, vz);
            else
                pp_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, px, py, pz, G, eps2, vx, vy, vz);
            rx = rx + vx; ry = ry + vy; rz = rz + vz;
        }
        const uint64_t open = mask & ~target_ballot<ROWS>(pass);
        if (open == 0) continue;
        const bool op = (open >> bit) & 1ull;
        if (nd.topo.z < 0) {
            const int first = nd.topo.x, cnt = nd.topo.y;
            if (first < 0 || cnt < 0 || (int64_t)first + cnt > a.n) { fail = true; break; }
            float lx, ly, lz;
            leaf_ordered<ROWS>(bodies, first, cnt, op, px, py, pz, G, eps2, lx, ly, lz);
            if (op) {
                cpp += (uint32_t)cnt;
                rx = rx + lx; ry = ry + ly; rz = rz + lz;
            }
        } else {
            if (sp + 3 > kStack || depth >= MAXD) { fail = true; break; }
            // pending depths ring_base .. depth - 1 are in the ring; a full
            // ring moves its shallowest level (all lanes) to scratch
            if (depth - ring_base >= RING) {
                const float *old = ring + (ring_base % RING) * 3 * kL + bit;
                s_save[ring_base * 3 + 0] = old[0];
                s_save[ring_base * 3 + 1] = old[kL];
                s_save[ring_base * 3 + 2] = old[2 * kL];
                ++ring_base;
            }
            if (op) {
                float *slot = ring + (depth % RING) * 3 * kL + bit;
                slot[0] = rx;
                slot[kL] = ry;
                slot[2 * kL] = rz;
                rx = 0.0f; ry = 0.0f; rz = 0.0f;
            }
            if (lane == 0) {
                s_node[sp] = node; s_meta[sp] = depth | kMetaComplete; s_mask[sp] = open;
                s_node[sp + 1] = nd.topo.z + 1; s_meta[sp + 1] = depth + 1; s_mask[sp + 1] = open;
                s_node[sp + 2] = nd.topo.z; s_meta[sp + 2] = depth + 1; s_mask[sp + 2] = open;
            }
            sp += 3;
        }
    }
}

// ORDERED linear-BVH walk, one wave per 64 targets from the root.
template <int MAXD, bool FOREST, bool QUAD>
__global__ __launch_bounds__(64 * kOrderedWaves) void k_walk_lbvh_ordered(WalkArgs a) {
    constexpr int kStack = 2 * MAXD + 4;
    __shared__ int s_node_all[kOrderedWaves][kStack];
    __shared__ int s_meta_all[kOrderedWaves][kStack];
    __shared__ uint64_t s_mask_all[kOrderedWaves][kStack];
    // Per lane, the pending partial sum of every open depth.  The pending
    // depths are those of the current path, saved in increasing depth and
    // taken back in decreasing depth, so the deepest kSaveRing of them live
    // in an LDS ring (slot d mod kSaveRing, lane-major: no bank conflicts)
    // and only older ones go to a private array indexed by the wave-uniform
    // depth (scratch memory): depths >= ring_base are in the ring.
    __shared__ float s_ring_all[kOrderedWaves][kSaveRing * 3 * kWave];

    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave);
    const WaveTask T = wave_task<FOREST>(a, (int64_t)walk_block<FOREST>() * kOrderedWaves + wv);
    const int64_t tgt = T.base + lane;
    const bool valid = tgt < T.end;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    uint32_t cpp = 0, cnp = 0;
    bool fail = false;
    ordered_descent<MAXD, QUAD, false, kSaveRing>(a, T.root, vmask, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv], s_meta_all[wv],
                                       s_mask_all[wv], s_ring_all[wv], rx, ry, rz, cpp, cnp, fail);
    if (fail && lane == 0) atomicOr(a.err, 2u);
    if (valid) {
        const uint32_t o = a.perm[tgt];
        if ((int64_t)o < a.nt) { a.ax[o] = rx; a.ay[o] = ry; a.az[o] = rz; }
    }
    const uint32_t wpp = wave_sum(valid ? cpp : 0u), wnp = wave_sum(valid ? cnp : 0u);
    if (lane == 0) {
        atomicAdd(&a.counts[0], (unsigned long long)wpp);
        atomicAdd(&a.counts[1], (unsigned long long)wnp);
    }
}

// ORDERED split (one linear BVH of middling size): a.split waves per group of
// 64 targets.  Each
// lists the frontier (the non-top children of opened top nodes, in the
// ORDERED walk's visit order, masks from the exact criterion), and wave k
// walks entries i with i mod a.split == k from zero, storing each subtree's
// result per target in split_part_f for k_walk_lbvh_ordered_combine.  Its
// frames would outgrow the LDS: by frames, 30,000 bodies (theta 0.5, leaf 64)
// took 2.80 ms to this walk's 2.32, 65,000 (leaf 16) 8.6 to 3.98.
template <int MAXD, bool QUAD>
__global__ __launch_bounds__(64 * kOrderedWaves) void k_walk_lbvh_ordered_split(WalkArgs a) {
    constexpr int kStack = 2 * MAXD + 4;
    __shared__ int s_node_all[kOrderedWaves][kStack];
    __shared__ int s_meta_all[kOrderedWaves][kStack];
    __shared__ uint64_t s_mask_all[kOrderedWaves][kStack];
    __shared__ float s_ring_all[kOrderedWaves][kSaveRing * 3 * kWave];
    __shared__ int f_node_all[kOrderedWaves][kMaxFrontier];
    __shared__ uint64_t f_mask_all[kOrderedWaves][kMaxFrontier];

    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave);
    const int K = a.split;
    const int64_t gw = (int64_t)xcd_block(blockIdx.x, gridDim.x) * kOrderedWaves + wv;
    const int64_t grp = gw / K;
    const int k = (int)(gw - grp * K);
    const WaveTask T = wave_task<false>(a, grp);
    const int64_t tgt = T.base + lane;
    const bool valid = tgt < T.end;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const NodeRec *__restrict__ nodes = a.nodes;
    int *s_node = s_node_all[wv];
    int *s_meta = s_meta_all[wv];
    uint64_t *s_mask = s_mask_all[wv];
    int *f_node = f_node_all[wv];
    uint64_t *f_mask = f_mask_all[wv];
    bool fail = false;

    // the frontier, in the order the ORDERED walk visits it
    const NodeRec root = nodes[T.root];
    const int cut = (root.topo.y + 31) / 32;
    int F = 0, sp = 1;
    if (lane == 0) { s_node[0] = T.root; s_meta[0] = 0; s_mask[0] = vmask; }
    __builtin_amdgcn_wave_barrier();
    while (sp > 0) {
        --sp;
        __builtin_amdgcn_wave_barrier();
        const int node = uniform_i32(s_node[sp]);
        const int depth = uniform_i32(s_meta[sp]);
        const uint64_t mask = uniform_u64(s_mask[sp]);
        if (node < 0 || node >= a.max_nodes) { fail = true; break; }
        const NodeRec nd = nodes[node];
        if (!lbvh_top(nd, depth, cut)) {
            if (F >= kMaxFrontier) { fail = true; break; }  // unreachable: depth <= kTopDepth
            if (lane == 0) { f_node[F] = node; f_mask[F] = mask; }
            ++F;
            continue;
        }
        const bool act = (mask >> lane) & 1ull;
        const uint64_t open = mask & ~__ballot(act && lbvh_accepts(nd.mac, me.x, me.y, me.z));
        if (open == 0) continue;
        if (sp + 2 > kStack) { fail = true; break; }
        if (lane == 0) {
            s_node[sp] = nd.topo.z + 1; s_meta[sp] = depth + 1; s_mask[sp] = open;
            s_node[sp + 1] = nd.topo.z; s_meta[sp + 1] = depth + 1; s_mask[sp + 1] = open;
        }
        __builtin_amdgcn_wave_barrier();
        sp += 2;
    }
    __builtin_amdgcn_wave_barrier();
    uint32_t cpp = 0, cnp = 0;
    const int64_t stride = a.split_stride;
    for (int i = k; i < F && !fail; i += K) {
        const int f = uniform_i32(f_node[i]);
        const uint64_t m = uniform_u64(f_mask[i]);
        float rx = 0.0f, ry = 0.0f, rz = 0.0f;
        ordered_descent<MAXD, QUAD, false, kSaveRing>(a, f, m, me.x, me.y, me.z, T.G, T.eps2, s_node, s_meta, s_mask,
                                           s_ring_all[wv], rx, ry, rz, cpp, cnp, fail);
        if (valid && ((m >> lane) & 1ull)) {
            const int64_t o = (int64_t)i * 3 * stride + tgt;
            a.split_part_f[o] = rx;
            a.split_part_f[o + stride] = ry;
            a.split_part_f[o + 2 * stride] = rz;
        }
    }
    if (fail && lane == 0) atomicOr(a.err, 2u);
    const uint32_t wpp = wave_sum(valid ? cpp : 0u), wnp = wave_sum(valid ? cnp : 0u);
    if (lane == 0) {
        atomicAdd(&a.counts[0], (unsigned long long)wpp);
        atomicAdd(&a.counts[1], (unsigned long long)wnp);
    }
}

// The ORDERED split's combine: the walk from the root over the top nodes,
// with each frontier subtree's stored result added where the walk meets it.
template <int MAXD, bool QUAD>
__global__ __launch_bounds__(64 * kOrderedWaves) void k_walk_lbvh_ordered_combine(WalkArgs a) {
    constexpr int kStack = 2 * MAXD + 4;
    __shared__ int s_node_all[kOrderedWaves][kStack];
    __shared__ int s_meta_all[kOrderedWaves][kStack];
    __shared__ uint64_t s_mask_all[kOrderedWaves][kStack];
    __shared__ float s_ring_all[kOrderedWaves][kSaveRing * 3 * kWave];

    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave);
    const WaveTask T = wave_task<false>(a, (int64_t)xcd_block(blockIdx.x, gridDim.x) * kOrderedWaves + wv);
    const int64_t tgt = T.base + lane;
    const bool valid = tgt < T.end;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const int cut = (a.nodes[T.root].topo.y + 31) / 32;
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    uint32_t cpp = 0, cnp = 0;
    bool fail = false;
    ordered_descent<MAXD, QUAD, false, kSaveRing, true>(a, T.root, vmask, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                      s_meta_all[wv], s_mask_all[wv], s_ring_all[wv], rx, ry, rz, cpp, cnp, fail,
                                      tgt, cut);
    if (fail && lane == 0) atomicOr(a.err, 2u);
    if (valid) {
        const uint32_t o = a.perm[tgt];
        if ((int64_t)o < a.nt) { a.ax[o] = rx; a.ay[o] = ry; a.az[o] = rz; }
    }
    const uint32_t wpp = wave_sum(valid ? cpp : 0u), wnp = wave_sum(valid ? cnp : 0u);
    if (lane == 0) {
        atomicAdd(&a.counts[0], (unsigned long long)wpp);
        atomicAdd(&a.counts[1], (unsigned long long)wnp);
    }
}

// The common end of a walk by frames: wave 0 holds the 16 targets' results
// (every row alike), the waves their counts (np: every row its own children;
// pp: every row the same leaves).
__device__ __forceinline__ void frames_end(const WalkArgs &a, int wv, int64_t tgt, bool valid, float rx, float ry,
                                           float rz, uint32_t cpp, uint32_t cnp, bool fail) {
    const int lane = lane_id();
    if (wv == 0 && valid && lane < kRowTargets) {
        const uint32_t o = a.perm[tgt];
        if ((int64_t)o < a.nt) { a.ax[o] = rx; a.ay[o] = ry; a.az[o] = rz; }
    }
    if (__ballot(fail) && lane == 0) atomicOr(a.err, 2u);
    const uint32_t wpp = wave_sum(lane < kRowTargets ? cpp : 0u), wnp = wave_sum(cnp);
    if (lane == 0) {
        if (wpp) atomicAdd(&a.counts[0], (unsigned long long)wpp);
        if (wnp) atomicAdd(&a.counts[1], (unsigned long long)wnp);
    }
}

// LDS writes of the wave's other lanes seen from here on.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The row's 16 bits of a ballot.
__device__ __forceinline__ uint32_t row_bits(uint64_t b, int row) { return (uint32_t)(b >> (16 * row)) & 0xFFFFu; }

// ORDERED linear-BVH walk by frames; a wave takes two frames at a time, one
// child per row.
template <int MAXD, bool QUAD, bool FOREST, int K>
__global__ __launch_bounds__(64 * K) void k_walk_lbvh_ordered_frames(WalkArgs a) {
    constexpr int kStack = 2 * MAXD + 4;
    constexpr int kSlots = frames_of(K, 16 * kStack + 4 * kRowsRing * 3 * kRowTargets);
    constexpr int kItems = items_of(K, kSlots), kFrames = kSlots - kItems;
    __shared__ int s_node_all[K][kStack];
    __shared__ int s_meta_all[K][kStack];
    __shared__ uint64_t s_mask_all[K][kStack];
    __shared__ float s_ring_all[K][kRowsRing * 3 * kRowTargets];
    __shared__ Frames<kSlots> F;

    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave), bit = target_bit<true>();
    const int row = lane / kRowTargets;
    const int64_t sub = walk_block<FOREST>();
    const WaveTask T = wave_task<FOREST>(a, sub / 4);
    const int64_t tgt = T.base + (sub % 4) * kRowTargets + bit;
    const bool valid = tgt < T.end;
    const uint64_t vmask = target_ballot<true>(valid);
    if (vmask == 0) return;  // the whole workgroup
    if (FOREST && (T.root < 0 || T.root >= a.max_nodes)) {  // no root was found: the whole workgroup
        if (threadIdx.x == 0) atomicOr(a.err, 2u);
        return;
    }
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const NodeRec *__restrict__ nodes = a.nodes;
    const float4 *__restrict__ bodies = a.bodies;
    bool fail = false;
    uint32_t cpp = 0, cnp = 0;

    // the root is a frame if a target opens it and it has children;
    // otherwise the walk ends with it
    const NodeRec rt = nodes[T.root];
    const uint32_t ropen = (uint32_t)vmask & ~(uint32_t)target_ballot<true>(valid && lbvh_accepts(rt.mac, me.x, me.y, me.z));
    const bool framed = ropen != 0 && rt.topo.z >= 0;
    if (threadIdx.x == 0) {
        F.tail = framed ? 1 : 0;
        F.itail = 0;
        F.next = 0;
        F.child[0] = rt.topo.z;
        F.mask[0] = (uint16_t)ropen;
    }
    __syncthreads();
    // levels: the level's frames are [lo, hi)
    int lo = 0, hi = framed ? 1 : 0, nlev = 0;
    while (lo < hi && nlev < MAXD && hi + 2 * (hi - lo) <= kFrames) {
        if (threadIdx.x == 0) F.first[nlev] = lo;
        ++nlev;
        for (int f2 = lo + 2 * wv; f2 < hi; f2 += 2 * K) {
            const int f = f2 + (row >> 1);
            const bool on = f < hi;
            const int c = on ? F.child[f] + (row & 1) : -1;
            const uint32_t O = on ? F.mask[f] : 0u;
            const bool ok = c >= 0 && c < a.max_nodes;
            if (on && !ok) fail = true;
            bool pass = false, inner = false;
            int down = -1;
            if (ok) {
                const NodeRec nd = nodes[c];
                pass = ((O >> bit) & 1u) && lbvh_accepts(nd.mac, me.x, me.y, me.z);
                inner = nd.topo.z >= 0;
                down = nd.topo.z;
            }
            const uint32_t open = O & ~row_bits(__ballot(pass), row);
            const bool kid = inner && open != 0;
            const uint64_t kb = __ballot(kid && bit == 0);  // one bit per row
            int base = 0;
            if (lane == 0 && kb) base = atomicAdd(&F.tail, __popcll(kb));
            base = uniform_i32(base);
            const uint64_t below = kb & ((1ull << (16 * row)) - 1);
            const int s = base + __popcll(below);
            if (kid && bit == 0) {
                F.child[s] = down;
                F.mask[s] = (uint16_t)open;
            }
            const uint64_t ib = kItems ? __ballot(ok && open != 0 && bit == 0 && !inner) : 0ull;
            int is = 0;
            if (lane == 0 && ib) is = atomicAdd(&F.itail, __popcll(ib));
            is = uniform_i32(is) + __popcll(ib & ((1ull << (16 * row)) - 1));
            if (((ib >> lane) & 1u) && is < kItems) {
                F.child[kFrames + is] = c;
                F.mask[kFrames + is] = (uint16_t)open;
            }
            if (on && (lane & 31) == 0) {
                F.slot[f] = (uint16_t)s;
                F.kids[f] = (uint16_t)(((kb >> (16 * row)) & 1u) | (((kb >> (16 * row + 16)) & 1u) << 1));
                F.islot[f] = (uint16_t)(is < kItems ? is : kItems);
                F.items[f] = (uint8_t)(((ib >> (16 * row)) & 1u) | (((ib >> (16 * row + 16)) & 1u) << 1));
            }
        }
        __syncthreads();
        lo = hi;
        hi = F.tail;
        __syncthreads();
    }
    // a last level too long for its children's slots, walked by the recursion,
    // and the listed leaves
    for (;;) {
        int i = 0;
        if (lane == 0) i = atomicAdd(&F.next, 1);
        i = uniform_i32(i);
        const bool deep = i < hi - lo;
        const int leaf = i - (hi - lo);
        if (!deep && (leaf >= kItems || leaf >= F.itail)) break;
        const int slot = deep ? lo + i : kFrames + leaf;
        const int c = uniform_i32(F.child[slot]);
        const uint32_t m = (uint32_t)uniform_i32((int)F.mask[slot]);
        float lx = 0.0f, ly = 0.0f, lz = 0.0f;
        if (deep) {
            uint32_t np = 0;
            for (int j = 0; j < 2; ++j)
                ordered_descent<MAXD, QUAD, true, kRowsRing>(a, c + j, m, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                                  s_meta_all[wv], s_mask_all[wv], s_ring_all[wv], lx, ly, lz, cpp, np,
                                                  fail);
            if (lane < kRowTargets) cnp += np;
        } else {
            const int4 topo = nodes[c].topo;
            const bool mine = (m >> bit) & 1u;
            if (topo.x < 0 || topo.y < 0 || (int64_t)topo.x + topo.y > a.n) { fail = true; continue; }
            leaf_ordered<true>(bodies, topo.x, topo.y, mine, me.x, me.y, me.z, T.G, T.eps2, lx, ly, lz);
            if (mine) cpp += (uint32_t)topo.y;
        }
        if (row == 0) {
            F.part[slot][0][bit] = lx;
            F.part[slot][1][bit] = ly;
            F.part[slot][2][bit] = lz;
        }
    }
    __syncthreads();
    // evaluation, from the last level up
    for (int lev = nlev - 1, end = lo; lev >= 0; --lev) {
        const int beg = uniform_i32(F.first[lev]);
        for (int f2 = beg + 2 * wv; f2 < end; f2 += 2 * K) {
            const int f = f2 + (row >> 1);
            const bool on = f < end;
            const int c = on ? F.child[f] + (row & 1) : -1;
            const uint32_t O = on ? F.mask[f] : 0u;
            const int kids = on ? F.kids[f] : 0, items = on ? F.items[f] : 0;
            // this child's slot, if it has one
            const int ks = on ? F.slot[f] + ((row & 1) ? (kids & 1) : 0) : 0;
            const int is = on ? F.islot[f] + ((row & 1) ? (items & 1) : 0) : 0;
            int from = -1;
            if ((kids >> (row & 1)) & 1) from = ks;
            if (((items >> (row & 1)) & 1) && is < kItems) from = kFrames + is;
            const bool ok = c >= 0 && c < a.max_nodes;
            NodeRec nd = {};
            if (ok) nd = nodes[c];
            const bool pass = ok && ((O >> bit) & 1u) && lbvh_accepts(nd.mac, me.x, me.y, me.z);
            float vx = 0.0f, vy = 0.0f, vz = 0.0f;
            if (pass) {
                ++cnp;
                if (QUAD)
                    np_quad_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, a.quad[2 * c], a.quad[2 * c + 1], me.x, me.y,
                                  me.z, T.G, T.eps2, vx, vy, vz);
                else
                    pp_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, me.x, me.y, me.z, T.G, T.eps2, vx, vy, vz);
            }
            const uint32_t open = ok ? O & ~row_bits(__ballot(pass), row) : 0u;
            const bool op = (open >> bit) & 1u;
            if (from >= 0 && op) {
                vx = F.part[from][0][bit];
                vy = F.part[from][1][bit];
                vz = F.part[from][2][bit];
            }
            // opened leaves that have no slot
            uint64_t rest = __ballot(open != 0 && bit == 0 && from < 0);
            while (rest) {
                const int l = __builtin_ctzll(rest);
                rest &= rest - 1;
                const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)open, l);
                const bool mine = (m >> bit) & 1u;
                float lx = 0.0f, ly = 0.0f, lz = 0.0f;
                const int first = __builtin_amdgcn_readlane(nd.topo.x, l), cnt = __builtin_amdgcn_readlane(nd.topo.y, l);
                if (first < 0 || cnt < 0 || (int64_t)first + cnt > a.n) { fail = true; continue; }
                leaf_ordered<true>(bodies, first, cnt, mine, me.x, me.y, me.z, T.G, T.eps2, lx, ly, lz);
                if (mine) cpp += (uint32_t)cnt;
                if (mine && row == l / kRowTargets) { vx = lx; vy = ly; vz = lz; }
            }
            // (0 + r0) + r1
            float x[4], y[4], z[4];
            spread_rows(vx, x);
            spread_rows(vy, y);
            spread_rows(vz, z);
            const bool second = row >= 2;
            const float Rx = (0.0f + (second ? x[2] : x[0])) + (second ? x[3] : x[1]);
            const float Ry = (0.0f + (second ? y[2] : y[0])) + (second ? y[3] : y[1]);
            const float Rz = (0.0f + (second ? z[2] : z[0])) + (second ? z[3] : z[1]);
            if (on && (row & 1) == 0) {
                F.part[f][0][bit] = Rx;
                F.part[f][1][bit] = Ry;
                F.part[f][2][bit] = Rz;
            }
        }
        end = beg;
        __syncthreads();
    }
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    if (wv == 0) {
        if (framed && ((ropen >> bit) & 1u)) {
            rx = F.part[0][0][bit];
            ry = F.part[0][1][bit];
            rz = F.part[0][2][bit];
        }
        // a root that is accepted, or a leaf
        const uint64_t m = framed ? vmask & ~(uint64_t)ropen : vmask;
        if (m) {
            float lx = 0.0f, ly = 0.0f, lz = 0.0f;
            uint32_t np = 0;
            ordered_descent<MAXD, QUAD, true, kRowsRing>(a, T.root, m, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv], s_meta_all[wv],
                                              s_mask_all[wv], s_ring_all[wv], lx, ly, lz, cpp, np, fail);
            if (lane < kRowTargets) cnp += np;
            if ((m >> bit) & 1ull) { rx = lx; ry = ly; rz = lz; }
        }
    }
    frames_end(a, wv, tgt, valid, rx, ry, rz, cpp, cnp, fail);
}

// ================================================================ octree
// ORDERED: libstdc++'s std::transform_reduce over the 8 children of an
// octree node (activeTree.h:66-76) computes init + ((r0 + r1) + (r2 + r3)),
// then + ((r4 + r5) + (r6 + r7)), with init = 0 and r = 0 for an empty
// child.  Per lane and per tree level the walk keeps that bracket's state
// in a private array (R: the running init, A: the open pair sum, B: the
// pending third term) and applies octant q's result with oct_step.
template <int MAXL>
__device__ __forceinline__ void oct_step(float *st, int q, bool act, float vx, float vy, float vz) {
    if (!act) return;
    float *R = st, *A = st + 3, *B = st + 6;
    const float v[3] = {vx, vy, vz};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int o = c;
        switch (q & 3) {
        case 0: A[o] = v[c]; break;
        case 1: A[o] = A[o] + v[c]; break;
        case 2: B[o] = v[c]; break;
        default: {
            const float a = A[o] + (B[o] + v[c]);
            A[o] = a;
            R[o] = q == 3 ? 0.0f + a : R[o] + a;
        }
        }
    }
}

// Evaluates node `nd` for the lanes in O: accepting lanes take its monopole
// and leaf lanes their leaf sum as this node's result r; returns the lanes
// that open it when it is internal.
// qn: the node's two moment records (QUAD only).
template <bool QUAD, bool ROWS>
__device__ __forceinline__ uint64_t oct_eval_ordered(const OctRec &nd, const float4 *__restrict__ qn, uint64_t O,
                                                     int bit, float px, float py, float pz, float G, float eps2,
                                                     const float4 *__restrict__ bodies, int64_t n, float &rx,
                                                     float &ry, float &rz, uint32_t &cpp, uint32_t &cnp, bool &fail) {
    const bool act = (O >> bit) & 1ull;
    const bool pass = act && oct_accepts(nd, px, py, pz);
    if (pass) {
        ++cnp;
        if (QUAD)
            np_quad_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, qn[0], qn[1], px, py, pz, G, eps2, rx, ry, rz);
        else
            pp_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, px, py, pz, G, eps2, rx, ry, rz);
    }
    const uint64_t open = O & ~target_ballot<ROWS>(pass);
    if (open == 0) return 0;
    if (nd.topo.z >= 0) return open;
    const int first = nd.topo.x, cnt = nd.topo.y;
    if (first < 0 || cnt < 0 || (int64_t)first + cnt > n) { fail = true; return 0; }
    const bool op = (open >> bit) & 1ull;
    float lx, ly, lz;
    leaf_ordered<ROWS>(bodies, first, cnt, op, px, py, pz, G, eps2, lx, ly, lz);
    if (op) {
        cpp += (uint32_t)cnt;
        rx = lx; ry = ly; rz = lz;
    }
    return 0;
}

// The ORDERED octree descent from node `start` for the lanes of `smask`: the
// node's result into r (assigned, as the reference's recursion returns it),
// counts into cpp / cnp.
template <int MAXL, bool QUAD, bool ROWS>
__device__ __forceinline__ void oct_ordered_descent(const WalkArgs &a, int start, uint64_t smask, float px, float py,
                                                    float pz, float G, float eps2, int *s_node, int *s_pos,
                                                    uint64_t *s_mask, float &rx, float &ry, float &rz, uint32_t &cpp,
                                                    uint32_t &cnp, bool &fail) {
    // Per lane and level, the bracket state (R, A, B; 3 floats each).  The
    // top frame's state lives in registers (cur); the frames below it are
    // parked in a private array indexed by the wave-uniform level (scratch
    // memory), written when a child is opened and read back when it
    // completes, so the child visits in between touch registers only.
    float s_st[MAXL * 9];
    float cur[9];
    const float4 *__restrict__ bodies = a.bodies;
    const OctRec *__restrict__ nodes = a.onodes;
    const int lane = lane_id(), bit = target_bit<ROWS>();
    int sp = 0;
    {
        const OctRec root = nodes[start];
        const uint64_t O = oct_eval_ordered<QUAD, ROWS>(root, a.quad + 2 * start, smask, bit, px, py, pz, G, eps2,
                                                  bodies, a.n, rx, ry, rz, cpp, cnp, fail);
        if (O) {
            if (lane == 0) { s_node[0] = start; s_pos[0] = 0; s_mask[0] = O; }
            sp = 1;
        }
    }
    // each frame is visited nchild + 1 <= 9 times, each node opened once
    const int64_t max_iters = 9 * a.max_nodes + 64;
    int64_t iters = 0;
    while (sp > 0 && !fail) {
        if (++iters > max_iters) { fail = true; break; }
        __builtin_amdgcn_wave_barrier();
        const int top = sp - 1;
        const int X = uniform_i32(s_node[top]);
        const int pos = uniform_i32(s_pos[top]);
        const uint64_t O = uniform_u64(s_mask[top]);
        const bool act = (O >> bit) & 1ull;
        if (X < 0 || X >= a.max_nodes) { fail = true; break; }
        const OctRec xr = nodes[X];
        const int cb = xr.topo.z, nch = oct_nchild(xr);
        if (cb < 0 || nch < 1 || nch > 8 || (int64_t)cb + nch > a.max_nodes) { fail = true; break; }
        int j = pos & 0xFF, q = pos >> 8;
        if (j > 0) {
            const int k = oct_octant(nodes[cb + j - 1]);
            for (; q < k; ++q) oct_step<MAXL>(cur, q, act, 0.0f, 0.0f, 0.0f);
            oct_step<MAXL>(cur, k, act, rx, ry, rz);
            q = k + 1;
        }
        if (j == nch) {
            for (; q < 8; ++q) oct_step<MAXL>(cur, q, act, 0.0f, 0.0f, 0.0f);
            if (act) { rx = cur[0]; ry = cur[1]; rz = cur[2]; }
            sp = top;
            if (top > 0) {  // the parent frame is the top again
#pragma unroll
                for (int i = 0; i < 9; ++i) cur[i] = s_st[(top - 1) * 9 + i];
            }
            continue;
        }
        if (lane == 0) s_pos[top] = (j + 1) | (q << 8);
        const OctRec cr = nodes[cb + j];
        const uint64_t open = oct_eval_ordered<QUAD, ROWS>(cr, a.quad + 2 * (cb + j), O, bit, px, py, pz, G, eps2, bodies,
                                                     a.n, rx, ry, rz, cpp, cnp, fail);
        if (open) {
            if (sp >= MAXL) { fail = true; break; }
            if (lane == 0) { s_node[sp] = cb + j; s_pos[sp] = 0; s_mask[sp] = open; }
            // park this frame's state; the child's frame starts in registers
            // (its first octant step writes before anything reads)
#pragma unroll
            for (int i = 0; i < 9; ++i) s_st[top * 9 + i] = cur[i];
            ++sp;
        }
    }
}

// The ORDERED octree walk, one wave per 64 targets from the root.
template <int MAXL, bool QUAD, bool FOREST>
__global__ __launch_bounds__(64 * kOrderedWaves) void k_walk_oct_ordered(WalkArgs a) {
    __shared__ int s_node_all[kOrderedWaves][MAXL];
    __shared__ int s_pos_all[kOrderedWaves][MAXL];  // next child index | next octant << 8
    __shared__ uint64_t s_mask_all[kOrderedWaves][MAXL];
    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave);
    const WaveTask T = wave_task<FOREST>(a, (int64_t)walk_block<FOREST>() * kOrderedWaves + wv);
    const int64_t tgt = T.base + lane;
    const bool valid = tgt < T.end;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    if (FOREST && (T.root < 0 || T.root >= a.max_nodes)) {
        if (lane == 0) atomicOr(a.err, 2u);
        return;
    }
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    uint32_t cpp = 0, cnp = 0;
    bool fail = false;
    oct_ordered_descent<MAXL, QUAD, false>(a, T.root, vmask, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                           s_pos_all[wv], s_mask_all[wv], rx, ry, rz, cpp, cnp, fail);
    if (fail && lane == 0) atomicOr(a.err, 2u);
    if (valid) {
        const uint32_t o = a.perm[tgt];
        if ((int64_t)o < a.nt) { a.ax[o] = rx; a.ay[o] = ry; a.az[o] = rz; }
    }
    const uint32_t wpp = wave_sum(valid ? cpp : 0u), wnp = wave_sum(valid ? cnp : 0u);
    if (lane == 0) {
        atomicAdd(&a.counts[0], (unsigned long long)wpp);
        atomicAdd(&a.counts[1], (unsigned long long)wnp);
    }
}

// ORDERED octree walk by frames; a wave takes one frame at a time, children j
// and j + 4 in row j.
template <int MAXL, bool QUAD, bool FOREST, int K>
__global__ __launch_bounds__(64 * K) void k_walk_oct_ordered_frames(WalkArgs a) {
    constexpr int kSlots = frames_of(K, 16 * MAXL + 4 * 8 * 3 * kRowTargets);
    constexpr int kItems = items_of(K, kSlots), kFrames = kSlots - kItems;
    __shared__ int s_node_all[K][MAXL];
    __shared__ int s_pos_all[K][MAXL];
    __shared__ uint64_t s_mask_all[K][MAXL];
    __shared__ float s_oct_all[K][8][3][kRowTargets];  // a frame's eight terms, on their way from rows to components
    __shared__ Frames<kSlots> F;

    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave), bit = target_bit<true>();
    const int row = lane / kRowTargets;
    const int64_t sub = walk_block<FOREST>();
    const WaveTask T = wave_task<FOREST>(a, sub / 4);
    const int64_t tgt = T.base + (sub % 4) * kRowTargets + bit;
    const bool valid = tgt < T.end;
    const uint64_t vmask = target_ballot<true>(valid);
    if (vmask == 0) return;  // the whole workgroup
    if (FOREST && (T.root < 0 || T.root >= a.max_nodes)) {  // no root was found: the whole workgroup
        if (threadIdx.x == 0) atomicOr(a.err, 2u);
        return;
    }
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const OctRec *__restrict__ nodes = a.onodes;
    const float4 *__restrict__ bodies = a.bodies;
    bool fail = false;
    uint32_t cpp = 0, cnp = 0;
    // children of a frame: count from kids' high bits
    auto kids_ok = [&](int cb, int nch) { return cb >= 0 && nch >= 1 && nch <= 8 && (int64_t)cb + nch <= a.max_nodes; };

    const OctRec rt = nodes[T.root];
    const uint32_t ropen = (uint32_t)vmask & ~(uint32_t)target_ballot<true>(valid && oct_accepts(rt, me.x, me.y, me.z));
    const bool framed = ropen != 0 && rt.topo.z >= 0;
    if (threadIdx.x == 0) {
        F.tail = framed ? 1 : 0;
        F.itail = 0;
        F.next = 0;
        F.child[0] = rt.topo.z;
        F.mask[0] = (uint16_t)ropen;
        F.kids[0] = (uint16_t)(oct_nchild(rt) << 8);
    }
    __syncthreads();
    int lo = 0, hi = framed ? 1 : 0, nlev = 0;
    while (lo < hi && nlev < MAXL) {
        if (threadIdx.x == 0) F.first[nlev] = lo;
        ++nlev;
        for (int f = lo + wv; f < hi; f += K) {
            const int cb = uniform_i32(F.child[f]);
            const uint32_t O = (uint32_t)uniform_i32((int)F.mask[f]);
            const int nch = uniform_i32((int)F.kids[f]) >> 8;
            if (!kids_ok(cb, nch)) { fail = true; if (lane == 0) F.kids[f] = 0; continue; }
            uint32_t open[2] = {0u, 0u};
            int down[2] = {-1, -1}, cnt[2] = {0, 0};
            uint32_t kids = 0, items = 0;
            // one bit per row
            auto per_row = [](uint64_t b) { return (uint32_t)((b & 1) | (b >> 15 & 2) | (b >> 30 & 4) | (b >> 45 & 8)); };
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (4 * h >= nch) break;
                const int j = row + 4 * h;
                bool pass = false;
                if (j < nch) {
                    const OctRec nd = nodes[cb + j];
                    pass = ((O >> bit) & 1u) && oct_accepts(nd, me.x, me.y, me.z);
                    down[h] = nd.topo.z;
                    cnt[h] = oct_nchild(nd);
                }
                const uint64_t pb = __ballot(pass);
                open[h] = j < nch ? O & ~row_bits(pb, row) : 0u;
                kids |= per_row(__ballot(open[h] != 0 && down[h] >= 0 && bit == 0)) << (4 * h);
                if (kItems) items |= per_row(__ballot(open[h] != 0 && down[h] < 0 && bit == 0)) << (4 * h);
            }
            int base = 0;
            if (lane == 0 && kids) base = atomicAdd(&F.tail, __popc(kids));
            base = uniform_i32(base);
            int ibase = 0;
            if (lane == 0 && items) ibase = atomicAdd(&F.itail, __popc(items));
            ibase = uniform_i32(ibase);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = row + 4 * h;
                const int s = base + __popc(kids & ((1u << j) - 1u));
                if (bit == 0 && ((kids >> j) & 1u) && s < kFrames) {
                    F.child[s] = down[h];
                    F.mask[s] = (uint16_t)open[h];
                    F.kids[s] = (uint16_t)(cnt[h] << 8);
                }
                const int is = ibase + __popc(items & ((1u << j) - 1u));
                if (bit == 0 && ((items >> j) & 1u) && is < kItems) {
                    F.child[kFrames + is] = cb + j;
                    F.mask[kFrames + is] = (uint16_t)open[h];
                }
            }
            if (lane == 0) {
                F.slot[f] = (uint16_t)(base < kFrames ? base : kFrames);
                F.kids[f] = (uint16_t)(kids | (nch << 8));
                F.islot[f] = (uint16_t)(ibase < kItems ? ibase : kItems);
                F.items[f] = (uint8_t)items;
            }
        }
        __syncthreads();
        lo = hi;
        hi = F.tail < kFrames ? F.tail : kFrames;
        __syncthreads();
    }
    if (lo < hi) { fail = true; nlev = 0; }  // deeper than any tree
    // the listed leaves
    if (kItems) {
        for (;;) {
            int i = 0;
            if (lane == 0) i = atomicAdd(&F.next, 1);
            i = uniform_i32(i);
            if (i >= kItems || i >= F.itail) break;
            const int4 topo = nodes[uniform_i32(F.child[kFrames + i])].topo;
            const bool mine = (F.mask[kFrames + i] >> bit) & 1u;
            float lx, ly, lz;
            if (topo.x < 0 || topo.y < 0 || (int64_t)topo.x + topo.y > a.n) { fail = true; continue; }
            leaf_ordered<true>(bodies, topo.x, topo.y, mine, me.x, me.y, me.z, T.G, T.eps2, lx, ly, lz);
            if (mine) cpp += (uint32_t)topo.y;
            if (row == 0) {
                F.part[kFrames + i][0][bit] = lx;
                F.part[kFrames + i][1][bit] = ly;
                F.part[kFrames + i][2][bit] = lz;
            }
        }
        __syncthreads();
    }
    float(*s_oct)[3][kRowTargets] = s_oct_all[wv];
    for (int lev = nlev - 1, end = lo; lev >= 0; --lev) {
        const int beg = uniform_i32(F.first[lev]);
        for (int f = beg + wv; f < end; f += K) {
            const int cb = uniform_i32(F.child[f]);
            const uint32_t O = (uint32_t)uniform_i32((int)F.mask[f]);
            const int kn = uniform_i32((int)F.kids[f]), slot = uniform_i32((int)F.slot[f]);
            const int nch = kn >> 8;
            const uint32_t kids = (uint32_t)kn & 0xFFu;
            const uint32_t items = (uint32_t)uniform_i32((int)F.items[f]);
            const int islot = uniform_i32((int)F.islot[f]);
            if (!kids_ok(cb, nch)) { fail = true; continue; }
            // absent octants count as zero
#pragma unroll
            for (int q = 0; q < 6; ++q) (&s_oct[0][0][0])[64 * q + lane] = 0.0f;
            wave_lds_fence();
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (4 * h >= nch) break;
                const int j = row + 4 * h;
                const bool on = j < nch;
                OctRec nd = {};
                nd.topo = make_int4(0, 0, -1, 0);
                if (on) nd = nodes[cb + j];
                const bool pass = on && ((O >> bit) & 1u) && oct_accepts(nd, me.x, me.y, me.z);
                float vx = 0.0f, vy = 0.0f, vz = 0.0f;
                if (pass) {
                    ++cnp;
                    if (QUAD)
                        np_quad_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, a.quad[2 * (cb + j)],
                                      a.quad[2 * (cb + j) + 1], me.x, me.y, me.z, T.G, T.eps2, vx, vy, vz);
                    else
                        pp_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, me.x, me.y, me.z, T.G, T.eps2, vx, vy, vz);
                }
                const uint64_t pb = __ballot(pass);
                const uint32_t open = on ? O & ~row_bits(pb, row) : 0u;
                const bool op = (open >> bit) & 1u;
                // this child's slot, if it has one
                const int ks = slot + __popc(kids & ((1u << j) - 1u)), is = islot + __popc(items & ((1u << j) - 1u));
                int from = -1;
                if (((kids >> j) & 1u) && ks < kFrames) from = ks;
                if (((items >> j) & 1u) && is < kItems) from = kFrames + is;
                if (from >= 0 && op) {
                    vx = F.part[from][0][bit];
                    vy = F.part[from][1][bit];
                    vz = F.part[from][2][bit];
                }
                // opened leaves and nodes that have no slot
                uint64_t rest = __ballot(open != 0 && bit == 0 && from < 0);
                while (rest) {
                    const int l = __builtin_ctzll(rest);
                    rest &= rest - 1;
                    const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)open, l);
                    const bool mine = (m >> bit) & 1u;
                    float lx = 0.0f, ly = 0.0f, lz = 0.0f;
                    if (__builtin_amdgcn_readlane(nd.topo.z, l) < 0) {
                        const int first = __builtin_amdgcn_readlane(nd.topo.x, l),
                                  cnt = __builtin_amdgcn_readlane(nd.topo.y, l);
                        if (first < 0 || cnt < 0 || (int64_t)first + cnt > a.n) { fail = true; continue; }
                        leaf_ordered<true>(bodies, first, cnt, mine, me.x, me.y, me.z, T.G, T.eps2, lx, ly, lz);
                        if (mine) cpp += (uint32_t)cnt;
                    } else {
                        uint32_t np = 0;
                        oct_ordered_descent<MAXL, QUAD, true>(a, cb + 4 * h + l / kRowTargets, m, me.x, me.y, me.z, T.G,
                                                              T.eps2, s_node_all[wv], s_pos_all[wv], s_mask_all[wv], lx,
                                                              ly, lz, cpp, np, fail);
                        if (lane < kRowTargets) cnp += np;
                    }
                    if (mine && row == l / kRowTargets) { vx = lx; vy = ly; vz = lz; }
                }
                if (on) {
                    const int q = oct_octant(nd) & 7;
                    s_oct[q][0][bit] = vx;
                    s_oct[q][1][bit] = vy;
                    s_oct[q][2][bit] = vz;
                }
            }
            wave_lds_fence();
            if (row < 3) {
                float v[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) v[q] = s_oct[q][row][bit];
                const float R = 0.0f + ((v[0] + v[1]) + (v[2] + v[3]));
                F.part[f][row][bit] = R + ((v[4] + v[5]) + (v[6] + v[7]));
            }
            wave_lds_fence();
        }
        end = beg;
        __syncthreads();
    }
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    if (wv == 0) {
        if (framed && nlev > 0 && ((ropen >> bit) & 1u)) {
            rx = F.part[0][0][bit];
            ry = F.part[0][1][bit];
            rz = F.part[0][2][bit];
        }
        // a root that is accepted, or a leaf
        const uint64_t m = framed ? vmask & ~(uint64_t)ropen : vmask;
        if (m) {
            float lx = 0.0f, ly = 0.0f, lz = 0.0f;
            uint32_t np = 0;
            oct_ordered_descent<MAXL, QUAD, true>(a, T.root, m, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                                  s_pos_all[wv], s_mask_all[wv], lx, ly, lz, cpp, np, fail);
            if (lane < kRowTargets) cnp += np;
            if ((m >> bit) & 1ull) { rx = lx; ry = ly; rz = lz; }
        }
    }
    frames_end(a, wv, tgt, valid, rx, ry, rz, cpp, cnp, fail);
}

// Waves the walk launches: one per 64 targets, or the forest's aligned waves.
static int64_t walk_waves(const WalkArgs &a) { return a.nsys > 0 ? a.nwaves : (a.nt + kWave - 1) / kWave; }

template <bool FOREST, bool QUAD, int MAXL>
static void launch_oct_frames_k(const WalkArgs &a, hipStream_t s) {
    const dim3 g((unsigned)(walk_waves(a) * 4));
    if (a.split >= 16) hipLaunchKernelGGL((k_walk_oct_ordered_frames<MAXL, QUAD, FOREST, 16>), g, dim3(1024), 0, s, a);
    else hipLaunchKernelGGL((k_walk_oct_ordered_frames<MAXL, QUAD, FOREST, 8>), g, dim3(512), 0, s, a);
}

template <bool FOREST>
static void launch_oct_frames(const WalkArgs &a, hipStream_t s) {
    const bool shallow = a.levels <= 18;
    if (a.quad && shallow) launch_oct_frames_k<FOREST, true, 18>(a, s);
    else if (a.quad) launch_oct_frames_k<FOREST, true, kOctLevels>(a, s);
    else if (shallow) launch_oct_frames_k<FOREST, false, 18>(a, s);
    else launch_oct_frames_k<FOREST, false, kOctLevels>(a, s);
}

template <int MAXD, bool FOREST, bool QUAD>
static void launch_lbvh_frames_k(const WalkArgs &a, hipStream_t s) {
    const dim3 g((unsigned)(walk_waves(a) * 4));
    if (a.split >= 16) hipLaunchKernelGGL((k_walk_lbvh_ordered_frames<MAXD, QUAD, FOREST, 16>), g, dim3(1024), 0, s, a);
    else hipLaunchKernelGGL((k_walk_lbvh_ordered_frames<MAXD, QUAD, FOREST, 8>), g, dim3(512), 0, s, a);
}

template <int MAXD, bool FOREST>
static void launch_lbvh_frames(const WalkArgs &a, hipStream_t s) {
    if (a.quad) launch_lbvh_frames_k<MAXD, FOREST, true>(a, s);
    else launch_lbvh_frames_k<MAXD, FOREST, false>(a, s);
}

void launch_walk_oct(const WalkArgs &a, int ordered, int stats, hipStream_t s) {
    if (a.n <= 0 || a.nt <= 0) return;
    if (!ordered) {
        launch_walk_fast(a, true, stats, s);
    } else if (a.split > 1) {
        if (a.nsys > 0) launch_oct_frames<true>(a, s);
        else launch_oct_frames<false>(a, s);
    } else {
        constexpr int W = kOrderedWaves;
        const unsigned blocks = (unsigned)((walk_waves(a) + W - 1) / W);
        const dim3 g(blocks), t(64 * W);
        const bool shallow = a.levels <= 18;  // a.levels: the deepest member's levels in a forest
        if (a.nsys > 0) {
            if (a.quad) {
                if (shallow) hipLaunchKernelGGL((k_walk_oct_ordered<18, true, true>), g, t, 0, s, a);
                else hipLaunchKernelGGL((k_walk_oct_ordered<kOctLevels, true, true>), g, t, 0, s, a);
            } else {
                if (shallow) hipLaunchKernelGGL((k_walk_oct_ordered<18, false, true>), g, t, 0, s, a);
                else hipLaunchKernelGGL((k_walk_oct_ordered<kOctLevels, false, true>), g, t, 0, s, a);
            }
        } else if (a.quad) {
            if (shallow) hipLaunchKernelGGL((k_walk_oct_ordered<18, true, false>), g, t, 0, s, a);
            else hipLaunchKernelGGL((k_walk_oct_ordered<kOctLevels, true, false>), g, t, 0, s, a);
        } else {
            if (shallow) hipLaunchKernelGGL((k_walk_oct_ordered<18, false, false>), g, t, 0, s, a);
            else hipLaunchKernelGGL((k_walk_oct_ordered<kOctLevels, false, false>), g, t, 0, s, a);
        }
    }
}

void launch_walk_lbvh(const WalkArgs &a, int ordered, int max_depth, int stats, hipStream_t s) {
    if (a.n <= 0 || a.nt <= 0) return;
    if (!ordered) {
        launch_walk_fast(a, false, stats, s);
    } else if (a.split_part_f) {
        constexpr int W = kOrderedWaves;
        const int64_t groups = (a.nt + kWave - 1) / kWave;
        const dim3 gs((unsigned)((groups * a.split + W - 1) / W)), gc((unsigned)((groups + W - 1) / W)), t(64 * W);
        if (a.quad && max_depth <= 32) {
            hipLaunchKernelGGL((k_walk_lbvh_ordered_split<32, true>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_lbvh_ordered_combine<32, true>), gc, t, 0, s, a);
        } else if (a.quad) {
            hipLaunchKernelGGL((k_walk_lbvh_ordered_split<64, true>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_lbvh_ordered_combine<64, true>), gc, t, 0, s, a);
        } else if (max_depth <= 32) {
            hipLaunchKernelGGL((k_walk_lbvh_ordered_split<32, false>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_lbvh_ordered_combine<32, false>), gc, t, 0, s, a);
        } else {
            hipLaunchKernelGGL((k_walk_lbvh_ordered_split<64, false>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_lbvh_ordered_combine<64, false>), gc, t, 0, s, a);
        }
    } else if (a.split > 1) {
        if (a.nsys > 0) launch_lbvh_frames<32, true>(a, s);
        else if (max_depth <= 32) launch_lbvh_frames<32, false>(a, s);
        else launch_lbvh_frames<64, false>(a, s);
    } else {
        constexpr int W = kOrderedWaves;
        const unsigned blocks = (unsigned)((walk_waves(a) + W - 1) / W);
        const dim3 g(blocks), t(64 * W);
        if (a.nsys > 0 && a.quad)
            hipLaunchKernelGGL((k_walk_lbvh_ordered<32, true, true>), g, t, 0, s, a);
        else if (a.nsys > 0)
            hipLaunchKernelGGL((k_walk_lbvh_ordered<32, true, false>), g, t, 0, s, a);
        else if (a.quad && max_depth <= 32)
            hipLaunchKernelGGL((k_walk_lbvh_ordered<32, false, true>), g, t, 0, s, a);
        else if (a.quad)
            hipLaunchKernelGGL((k_walk_lbvh_ordered<64, false, true>), g, t, 0, s, a);
        else if (max_depth <= 32)
            hipLaunchKernelGGL((k_walk_lbvh_ordered<32, false, false>), g, t, 0, s, a);
        else
            hipLaunchKernelGGL((k_walk_lbvh_ordered<64, false, false>), g, t, 0, s, a);
    }
}

}  // namespace nbg
