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
// on where it is computed, so a small system's walk can be split: frontier
// subtrees walked from zero by several waves, their results used where the
// walk over the top nodes meets them, with unchanged bits.
//
// The FAST walks (walk_fast.hip) take the same opening decisions in another
// schedule.

#include "device.hpp"
#include "launch.hpp"
#include "walk_common.hpp"
#include "walk_task.hpp"

namespace nbg {

constexpr int kMetaComplete = 0x10000;
// Upper bound on loop iterations per wave; a valid tree needs at most ~3 per node.
constexpr uint32_t kMaxWalkIters = 1u << 28;

// The top of a linear BVH, for the split walks: internal nodes above
// depth kTopDepth holding more than `cut` bodies.  Their other children are
// the frontier, at most 2^kTopDepth nodes.
constexpr int kTopDepth = 7;
constexpr int kMaxFrontier = 1 << kTopDepth;
static_assert(kMaxFrontier == kOrderedSplitSlots, "ORDERED split: one slot per frontier entry");

__device__ __forceinline__ bool lbvh_top(const NodeRec &r, int depth, int cut) {
    return r.topo.z >= 0 && r.topo.y > cut && depth < kTopDepth;
}

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

// Levels of pending partial sums an ORDERED linear-BVH wave keeps in LDS.
constexpr int kSaveRing = 4;

// The ORDERED descent from node `start` for the lanes of `smask`, the
// reference's recursion (activeTree.h:24-79) with its bracketing: each node's
// result into r (from zero), counts into cpp / cnp.  COMBINE: a visited node
// that is not a top node (lbvh_top with the root's cut) is a frontier node:
// its result is not walked but taken from part (slot fi, counted in visit
// order) and added as the walk would add it.
template <int MAXD, bool QUAD, bool COMBINE>
__device__ __forceinline__ void ordered_descent(const WalkArgs &a, int start, uint64_t smask, int cut, float px,
                                                float py, float pz, float G, float eps2, int *s_node, int *s_meta,
                                                uint64_t *s_mask, float *ring, float &rx, float &ry, float &rz,
                                                uint32_t &cpp, uint32_t &cnp, bool &fail, int64_t tgt) {
    constexpr int kStack = 2 * MAXD + 4;
    float s_save[MAXD * 3];
    const float4 *__restrict__ bodies = a.bodies;
    const NodeRec *__restrict__ nodes = a.nodes;
    const int lane = lane_id();
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
        const bool act = (mask >> lane) & 1ull;
        const int depth = meta & 0xFFFF;
        if (meta & kMetaComplete) {
            // the deepest pending depth comes back: from the ring, or (the
            // ring then holds nothing) from scratch
            if (depth >= ring_base) {
                const float *slot = ring + (depth % kSaveRing) * 3 * kWave + lane;
                if (act) {
                    const float vx = rx, vy = ry, vz = rz;
                    rx = slot[0] + vx;
                    ry = slot[kWave] + vy;
                    rz = slot[2 * kWave] + vz;
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
        if (COMBINE && !lbvh_top(nd, depth, cut)) {
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
        const uint64_t open = mask & ~__ballot(pass);
        if (open == 0) continue;
        const bool op = (open >> lane) & 1ull;
        if (nd.topo.z < 0) {
            const int first = nd.topo.x, cnt = nd.topo.y;
            if (first < 0 || cnt < 0 || (int64_t)first + cnt > a.n) { fail = true; break; }
            // the body loop runs in wave-uniform flow so its loads are scalar
            // (one per body for the wave); the opened lanes sum
            float lx = 0.0f, ly = 0.0f, lz = 0.0f;
            for (int j = 0; j < cnt; ++j) {
                const float4 b = bodies[first + j];
                if (op) {
                    float vx, vy, vz;
                    pp_exact(b.x, b.y, b.z, b.w, px, py, pz, G, eps2, vx, vy, vz);
                    lx = lx + vx; ly = ly + vy; lz = lz + vz;
                }
            }
            if (op) {
                cpp += (uint32_t)cnt;
                rx = rx + lx; ry = ry + ly; rz = rz + lz;
            }
        } else {
            if (sp + 3 > kStack || depth >= MAXD) { fail = true; break; }
            // pending depths ring_base .. depth - 1 are in the ring; a full
            // ring moves its shallowest level (all lanes) to scratch
            if (depth - ring_base >= kSaveRing) {
                const float *old = ring + (ring_base % kSaveRing) * 3 * kWave + lane;
                s_save[ring_base * 3 + 0] = old[0];
                s_save[ring_base * 3 + 1] = old[kWave];
                s_save[ring_base * 3 + 2] = old[2 * kWave];
                ++ring_base;
            }
            if (op) {
                float *slot = ring + (depth % kSaveRing) * 3 * kWave + lane;
                slot[0] = rx;
                slot[kWave] = ry;
                slot[2 * kWave] = rz;
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
    const WaveTask T = wave_task<FOREST>(a, (int64_t)xcd_block(blockIdx.x, gridDim.x) * kOrderedWaves + wv);
    const int64_t tgt = T.base + lane;
    const bool valid = tgt < T.end;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    uint32_t cpp = 0, cnp = 0;
    bool fail = false;
    ordered_descent<MAXD, QUAD, false>(a, T.root, vmask, 0, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                       s_meta_all[wv], s_mask_all[wv], s_ring_all[wv], rx, ry, rz, cpp, cnp, fail,
                                       tgt);
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

// ORDERED split (one system): a.split waves per group of 64 targets.  Each
// lists the frontier (the non-top children of opened top nodes, in the
// ORDERED walk's visit order, masks from the exact criterion), and wave k
// walks entries i with i mod a.split == k from zero, storing each subtree's
// result per target in split_part_f for k_walk_lbvh_ordered_combine.
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
        ordered_descent<MAXD, QUAD, false>(a, f, m, cut, me.x, me.y, me.z, T.G, T.eps2, s_node, s_meta, s_mask,
                                           s_ring_all[wv], rx, ry, rz, cpp, cnp, fail, tgt);
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
    ordered_descent<MAXD, QUAD, true>(a, T.root, vmask, cut, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                      s_meta_all[wv], s_mask_all[wv], s_ring_all[wv], rx, ry, rz, cpp, cnp, fail,
                                      tgt);
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
template <bool QUAD>
__device__ __forceinline__ uint64_t oct_eval_ordered(const OctRec &nd, const float4 *__restrict__ qn, uint64_t O,
                                                     int lane, float px, float py, float pz, float G, float eps2,
                                                     const float4 *__restrict__ bodies, int64_t n, float &rx,
                                                     float &ry, float &rz, uint32_t &cpp, uint32_t &cnp, bool &fail) {
    const bool act = (O >> lane) & 1ull;
    const bool pass = act && oct_accepts(nd, px, py, pz);
    if (pass) {
        ++cnp;
        if (QUAD)
            np_quad_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, qn[0], qn[1], px, py, pz, G, eps2, rx, ry, rz);
        else
            pp_exact(nd.com.x, nd.com.y, nd.com.z, nd.com.w, px, py, pz, G, eps2, rx, ry, rz);
    }
    const uint64_t open = O & ~__ballot(pass);
    if (open == 0) return 0;
    if (nd.topo.z >= 0) return open;
    const int first = nd.topo.x, cnt = nd.topo.y;
    if (first < 0 || cnt < 0 || (int64_t)first + cnt > n) { fail = true; return 0; }
    // the body loop runs in wave-uniform flow so its loads are scalar
    const bool op = (open >> lane) & 1ull;
    float lx = 0.0f, ly = 0.0f, lz = 0.0f;
    for (int j = 0; j < cnt; ++j) {
        const float4 b = bodies[first + j];
        if (op) {
            float vx, vy, vz;
            pp_exact(b.x, b.y, b.z, b.w, px, py, pz, G, eps2, vx, vy, vz);
            lx = lx + vx; ly = ly + vy; lz = lz + vz;
        }
    }
    if (op) {
        cpp += (uint32_t)cnt;
        rx = lx; ry = ly; rz = lz;
    }
    return 0;
}

// The top of an octree for the ORDERED split: internal nodes at depth 0 or 1
// holding more than `cut` bodies.  Their other children are the frontier
// (at most 8 + 64 nodes).
__device__ __forceinline__ bool oct_top_ordered(const OctRec &r, int depth, int cut) {
    return r.topo.z >= 0 && r.topo.y > cut && depth < 2;
}

// The ORDERED octree descent from node `start` for the lanes of `smask`: the
// node's result into r (assigned, as the reference's recursion returns it),
// counts into cpp / cnp.  COMBINE: a child that is not a top node (with the
// root's cut) is a frontier node: its result is taken from split_part_f
// (slot fi, counted in visit order) instead of being evaluated.
template <int MAXL, bool QUAD, bool COMBINE>
__device__ __forceinline__ void oct_ordered_descent(const WalkArgs &a, int start, uint64_t smask, int cut, float px,
                                                    float py, float pz, float G, float eps2, int *s_node, int *s_pos,
                                                    uint64_t *s_mask, float &rx, float &ry, float &rz, uint32_t &cpp,
                                                    uint32_t &cnp, bool &fail, int64_t tgt) {
    // Per lane and level, the bracket state (R, A, B; 3 floats each).  The
    // top frame's state lives in registers (cur); the frames below it are
    // parked in a private array indexed by the wave-uniform level (scratch
    // memory), written when a child is opened and read back when it
    // completes, so the child visits in between touch registers only.
    float s_st[MAXL * 9];
    float cur[9];
    const float4 *__restrict__ bodies = a.bodies;
    const OctRec *__restrict__ nodes = a.onodes;
    const int lane = lane_id();
    int fi = 0;
    auto frontier = [&](uint64_t O) {
        if (fi >= kOrderedSplitSlots) { fail = true; return; }
        if ((O >> lane) & 1ull) {
            const int64_t o = (int64_t)fi * 3 * a.split_stride + tgt;
            rx = a.split_part_f[o];
            ry = a.split_part_f[o + a.split_stride];
            rz = a.split_part_f[o + 2 * a.split_stride];
        }
        ++fi;
    };
    int sp = 0;
    {
        const OctRec root = nodes[start];
        if (COMBINE && !oct_top_ordered(root, 0, cut)) {
            frontier(smask);
            return;
        }
        const uint64_t O = oct_eval_ordered<QUAD>(root, a.quad + 2 * start, smask, lane, px, py, pz, G, eps2,
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
        const bool act = (O >> lane) & 1ull;
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
        if (COMBINE && !oct_top_ordered(cr, top + 1, cut)) {
            frontier(O);
            continue;
        }
        const uint64_t open = oct_eval_ordered<QUAD>(cr, a.quad + 2 * (cb + j), O, lane, px, py, pz, G, eps2, bodies,
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
    const WaveTask T = wave_task<FOREST>(a, (int64_t)xcd_block(blockIdx.x, gridDim.x) * kOrderedWaves + wv);
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
    oct_ordered_descent<MAXL, QUAD, false>(a, T.root, vmask, 0, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                           s_pos_all[wv], s_mask_all[wv], rx, ry, rz, cpp, cnp, fail, tgt);
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

// ORDERED octree split (one system): a.split waves per group of 64 targets.
// Each lists the frontier in the ORDERED walk's visit order (masks: the lanes
// that evaluate the node), and wave k computes the results of entries
// i with i mod a.split == k, as the walk would (each node's result is
// assigned, not accumulated), for k_walk_oct_ordered_combine.
template <int MAXL, bool QUAD>
__global__ __launch_bounds__(64 * kOrderedWaves) void k_walk_oct_ordered_split(WalkArgs a) {
    __shared__ int s_node_all[kOrderedWaves][MAXL];
    __shared__ int s_pos_all[kOrderedWaves][MAXL];
    __shared__ uint64_t s_mask_all[kOrderedWaves][MAXL];
    __shared__ int f_node_all[kOrderedWaves][kOrderedSplitSlots];
    __shared__ uint64_t f_mask_all[kOrderedWaves][kOrderedSplitSlots];
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
    const OctRec *__restrict__ nodes = a.onodes;
    int *s_node = s_node_all[wv];
    int *s_pos = s_pos_all[wv];
    uint64_t *s_mask = s_mask_all[wv];
    int *f_node = f_node_all[wv];
    uint64_t *f_mask = f_mask_all[wv];
    bool fail = false;

    // the frontier, in the order the ORDERED walk meets it: frames over the
    // top nodes, children in index order, a top child's frame walked before
    // its later siblings
    const OctRec root = nodes[T.root];
    const int cut = (root.topo.y + 31) / 32;
    int F = 0, sp = 0;
    auto add = [&](int node, uint64_t m) {
        if (F >= kOrderedSplitSlots) { fail = true; return; }
        if (lane == 0) { f_node[F] = node; f_mask[F] = m; }
        ++F;
    };
    if (!oct_top_ordered(root, 0, cut)) {
        add(T.root, vmask);
    } else {
        const bool act = (vmask >> lane) & 1ull;
        const uint64_t O = vmask & ~__ballot(act && oct_accepts(root, me.x, me.y, me.z));
        if (O) {
            if (lane == 0) { s_node[0] = T.root; s_pos[0] = 0; s_mask[0] = O; }
            sp = 1;
        }
    }
    while (sp > 0 && !fail) {
        __builtin_amdgcn_wave_barrier();
        const int top = sp - 1;
        const int X = uniform_i32(s_node[top]);
        const int j = uniform_i32(s_pos[top]);
        const uint64_t O = uniform_u64(s_mask[top]);
        if (X < 0 || X >= a.max_nodes) { fail = true; break; }
        const OctRec xr = nodes[X];
        const int cb = xr.topo.z, nch = oct_nchild(xr);
        if (cb < 0 || nch < 1 || nch > 8 || (int64_t)cb + nch > a.max_nodes) { fail = true; break; }
        if (j == nch) {
            sp = top;
            continue;
        }
        if (lane == 0) s_pos[top] = j + 1;
        const OctRec cr = nodes[cb + j];
        if (!oct_top_ordered(cr, top + 1, cut)) {
            add(cb + j, O);
            continue;
        }
        const bool act = (O >> lane) & 1ull;
        const uint64_t open = O & ~__ballot(act && oct_accepts(cr, me.x, me.y, me.z));
        if (open) {
            if (sp >= MAXL) { fail = true; break; }
            if (lane == 0) { s_node[sp] = cb + j; s_pos[sp] = 0; s_mask[sp] = open; }
            ++sp;
        }
    }
    __builtin_amdgcn_wave_barrier();
    uint32_t cpp = 0, cnp = 0;
    const int64_t stride = a.split_stride;
    for (int i = k; i < F && !fail; i += K) {
        const int f = uniform_i32(f_node[i]);
        const uint64_t m = uniform_u64(f_mask[i]);
        float rx = 0.0f, ry = 0.0f, rz = 0.0f;
        oct_ordered_descent<MAXL, QUAD, false>(a, f, m, cut, me.x, me.y, me.z, T.G, T.eps2, s_node, s_pos, s_mask, rx,
                                               ry, rz, cpp, cnp, fail, tgt);
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

// The ORDERED octree split's combine: the walk over the top nodes, each
// frontier child's stored result applied to its parent's bracket.
template <int MAXL, bool QUAD>
__global__ __launch_bounds__(64 * kOrderedWaves) void k_walk_oct_ordered_combine(WalkArgs a) {
    __shared__ int s_node_all[kOrderedWaves][MAXL];
    __shared__ int s_pos_all[kOrderedWaves][MAXL];
    __shared__ uint64_t s_mask_all[kOrderedWaves][MAXL];
    const int lane = lane_id(), wv = uniform_i32(threadIdx.x / kWave);
    const WaveTask T = wave_task<false>(a, (int64_t)xcd_block(blockIdx.x, gridDim.x) * kOrderedWaves + wv);
    const int64_t tgt = T.base + lane;
    const bool valid = tgt < T.end;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    const float4 me = valid ? a.targets[tgt] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const int cut = (a.onodes[T.root].topo.y + 31) / 32;
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    uint32_t cpp = 0, cnp = 0;
    bool fail = false;
    oct_ordered_descent<MAXL, QUAD, true>(a, T.root, vmask, cut, me.x, me.y, me.z, T.G, T.eps2, s_node_all[wv],
                                          s_pos_all[wv], s_mask_all[wv], rx, ry, rz, cpp, cnp, fail, tgt);
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

// Waves the walk launches: one per 64 targets, or the forest's aligned waves.
static int64_t walk_waves(const WalkArgs &a) { return a.nsys > 0 ? a.nwaves : (a.nt + kWave - 1) / kWave; }

void launch_walk_oct(const WalkArgs &a, int ordered, int stats, hipStream_t s) {
    if (a.n <= 0 || a.nt <= 0) return;
    if (!ordered) {
        launch_walk_fast(a, true, stats, s);
    } else if (a.nsys == 0 && a.split > 1 && a.split_part_f) {
        constexpr int W = kOrderedWaves;
        const int64_t groups = (a.nt + kWave - 1) / kWave;
        const dim3 gs((unsigned)((groups * a.split + W - 1) / W)), gc((unsigned)((groups + W - 1) / W)), t(64 * W);
        const bool shallow = a.levels <= 18;
        if (a.quad && shallow) {
            hipLaunchKernelGGL((k_walk_oct_ordered_split<18, true>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_oct_ordered_combine<18, true>), gc, t, 0, s, a);
        } else if (a.quad) {
            hipLaunchKernelGGL((k_walk_oct_ordered_split<kOctLevels, true>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_oct_ordered_combine<kOctLevels, true>), gc, t, 0, s, a);
        } else if (shallow) {
            hipLaunchKernelGGL((k_walk_oct_ordered_split<18, false>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_oct_ordered_combine<18, false>), gc, t, 0, s, a);
        } else {
            hipLaunchKernelGGL((k_walk_oct_ordered_split<kOctLevels, false>), gs, t, 0, s, a);
            hipLaunchKernelGGL((k_walk_oct_ordered_combine<kOctLevels, false>), gc, t, 0, s, a);
        }
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
    } else if (a.nsys == 0 && a.split > 1 && a.split_part_f) {
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
