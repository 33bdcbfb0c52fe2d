// FAST Barnes-Hut walks for gfx950 (linear BVH and octree, monopole and
// quadrupole, one system or a forest).
//
// One wavefront walks the tree for kSub = 16 spatially adjacent targets.  It
// works in two alternating phases, each with all 64 lanes busy:
//
//   listing: lane = tree node.  A node waits on an LDS stack with the mask of
//     the targets that reached it.  Its opening test is first taken against
//     the targets' bounding box: a node that every point of the box accepts
//     goes to the interaction list with its mask, one that every point
//     rejects is opened with its mask.  Both bounds go through the criterion's
//     own FP32 operations in its own order, and rounding is monotone, so they
//     decide exactly as the targets would.  The other nodes wait in a queue,
//     and 64 at a time take the criterion of each target in turn (targets in
//     scalar registers), which splits their masks.  Opened internal nodes go
//     back to the stack, bodies of opened leaves to the interaction list.
//   summing: lane = (target, row).  The list's 64 sources are taken four at a
//     time, one per 16-lane row, each lane adding its row's source to its
//     target's sum; the rows meet once, at the end of the walk.
//
// Each target meets exactly the nodes and bodies that the reference's
// per-body recursion meets (Descent/activeTree.h:24-79).
//
// Why: a wavefront that visits each node with 64 targets in its lanes spends
// 9 instructions a node on tests that are unanimous for half of the nodes,
// and 13 on interactions that 46 % (nodes) and 62 % (leaf bodies) of its
// lanes mask out (1,048,576 Plummer bodies, theta 0.5, linear BVH), and each
// visit waits for the one before it.  Sixteen targets leave 31 % and 44 % of
// the lanes masked out, 64 unanimous tests take about 100 instructions, and
// the sources of a list do not depend on each other: 13 instructions for 64
// of them, 15 with masks.  Measured against that walk, ms a pass: linear BVH
// 7.71 -> 5.20, octree 3.74 -> 2.05 (1,048,576 bodies), quadrupole linear
// BVH 2.51 -> 1.90 (500,000), octree 2.58 -> 1.54 (300,007, theta 0.41),
// linear BVH of 10,000 bodies 0.41 -> 0.14.  Bound by VALU issue (linear BVH,
// targets in compact groups: 43,100 instructions a wave and 65,536 waves are
// 4.6 ms at 2.4 GHz on 1,024 SIMDs), of which the pairs' own are 35 %; half
// the targets a wave would double the listing.
//
// Sums: the 64 sources of a list are four classes of 16; each class has its
// own FP32 partial per lane (at most 32 terms, then added to FP64), and the
// result is ((c0 + c1) + (c2 + c3)) over the classes' row sums in FP64, times
// G, rounded once.  The K waves of a small system's group all list, and each
// sums its share of the classes, so the bits do not depend on K.

#include <type_traits>

#include "device.hpp"
#include "launch.hpp"
#include "walk_common.hpp"
#include "walk_task.hpp"

namespace nbg {

constexpr int kSub = 16;                  // targets per wave
constexpr int kRows = kWave / kSub;       // sources a wave sums at once
constexpr int kFastWaves = 4;             // waves per workgroup
constexpr int kClasses = 4;               // independent sums of a target
constexpr int kFlushEvery = 8;            // lists of 64 between additions to FP64 (32 terms per lane and class)
// The list of sources that every target takes grows up from the buffer's
// start, the one of sources with a mask down from its end.  Each is summed as
// soon as it holds 64, and one step adds at most 64 to both together.
constexpr int kListCap = 3 * kWave;
constexpr int kMaskCap = 2 * kWave;       // entries of a list with masks
constexpr int kMixCap = 2 * kWave;
constexpr int kLeafKeep = 15;              // leaves are expanded while more wait
constexpr int kLeafCap = kWave + kLeafKeep;  // leaves of one step: at most 64
constexpr uint32_t kMaxFastIters = 1u << 28;

// The stack holds sibling groups (first child, mask).  Steps pop up to 64
// lanes' worth of groups while the stack stays within kWide groups, and one
// group at a time where it would not, so the stack never outgrows kWide + 64
// (queued mixed nodes) plus the growth of a depth-first descent (1 or 7
// groups a level).  kWide is what full steps need at theta 0.3 and below on
// 1,048,576 bodies (linear BVH: 281 groups on average, 512 at most; octree
// 136 and 206) as far as the LDS of four workgroups a CU holds it, three for
// the quadrupoles: with 128 groups the linear BVH's steps degenerate to one
// group and its walk of 1,048,576 bodies took 24.8 ms.
constexpr int wide_groups(bool oct, bool quad) { return oct ? (quad ? 176 : 256) : (quad ? 392 : 512); }
constexpr int stack_groups(bool oct, bool quad) {
    return wide_groups(oct, quad) + kWave + (oct ? 8 * (kOctLevels + 2) : 72);  // a linear BVH has at most 64 levels
}

template <bool OCT, bool QUAD>
struct WaveLds {
    static constexpr int kStack = stack_groups(OCT, QUAD);
    float4 src[QUAD ? kMaskCap : kListCap];  // QUAD: bodies only, all with masks
    float4 qsrc[QUAD ? 3 : 1][QUAD ? kMaskCap : 1];  // QUAD: accepted nodes' centres of mass and moments
    int st_node[kStack];
    int mq_node[kMixCap];
    int lq_first[kLeafCap], lq_cnt[kLeafCap];
    uint16_t st_mask[kStack];
    uint16_t mq_mask[kMixCap];
    uint16_t lq_mask[kLeafCap];
    uint16_t smask[kMaskCap];                // masks of src[end - 1 - e]
    uint16_t qmask[QUAD ? kMaskCap : 1];
    uint32_t starts[2];                      // lanes at which a leaf's bodies start
};

// Orders this wave's LDS writes and reads among its lanes (the hardware keeps
// a wave's LDS operations in order; this holds the compiler to it).
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int rank_in(uint64_t b) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
}

__device__ __forceinline__ bool in_lane(uint64_t b) { return __builtin_amdgcn_inverse_ballot_w64(b); }

__device__ __forceinline__ uint64_t lanes_below(int n) { return n >= kWave ? ~0ull : (1ull << n) - 1ull; }

// Inclusive scan over the wave, in the vector unit (row shifts, then the rows'
// last lanes broadcast to the rows after them).
__device__ __forceinline__ int incl_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 to rows 2 and 3
    return v;
}

// 2 v + (this lane's bit of b), in one instruction.
__device__ __forceinline__ uint32_t shift_in(uint32_t v, uint64_t b) {
    uint64_t carry;
    asm("v_addc_co_u32_e64 %0, %1, %2, %2, %3" : "=v"(v), "=s"(carry) : "v"(v), "s"(b));
    return v;
}

struct Pair3 {
    float x, y, z;
};

// One source into a lane's partial sum; bits: all ones, or zero to leave the
// lane out (the scale is cleared, so nothing of a left-out lane's distance
// reaches its sum).
template <bool SOFT, bool MASKED>
__device__ __forceinline__ void add_source(float4 b, uint32_t bits, float px, float py, float pz, float eps2, Pair3 &r) {
    const float dx = b.x - px, dy = b.y - py, dz = b.z - pz;
    const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, eps2)));
    float inv = __builtin_amdgcn_rsqf(r2);
    if (!SOFT) inv = r2 > 0.0f ? inv : 0.0f;
    float s = b.w * (inv * (inv * inv));
    if (MASKED) s = __uint_as_float(__float_as_uint(s) & bits);
    r.x = __builtin_fmaf(dx, s, r.x);
    r.y = __builtin_fmaf(dy, s, r.y);
    r.z = __builtin_fmaf(dz, s, r.z);
}

// Quadrupole node interaction (Gravity::nodeParticle<2>, Gravity.h:238-259)
// with rsqrt + FMA.  With d = c - p (the reference's R = -d), the reference's
// R (-M) / r^3 + D3(R) . Q / 2 expands to
//   d (M r^-3 + 7.5 r^-7 d.Q.d - 1.5 r^-5 tr Q) - 3 r^-5 Q d,
// r^2 = d.d + eps2; G is applied once at the end of the walk.  d = 0 (the
// target at the node's COM) contributes exactly zero.
template <bool SOFT>
__device__ __forceinline__ void add_quad(float4 b, float4 q0, float4 q1, uint32_t bits, float px, float py, float pz,
                                         float eps2, Pair3 &r) {
    const float dx = b.x - px, dy = b.y - py, dz = b.z - pz;
    const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, eps2)));
    float inv = __builtin_amdgcn_rsqf(r2);
    if (!SOFT) inv = r2 > 0.0f ? inv : 0.0f;
    const float inv2 = inv * inv, inv3 = inv * inv2, inv5 = inv3 * inv2;
    // Q d with Q = [[xx xy xz] [xy yy yz] [xz yz zz]] = [[q0.x q0.y q0.z] [q0.y q0.w q1.x] [q0.z q1.x q1.y]]
    const float qx = __builtin_fmaf(q0.x, dx, __builtin_fmaf(q0.y, dy, q0.z * dz));
    const float qy = __builtin_fmaf(q0.y, dx, __builtin_fmaf(q0.w, dy, q1.x * dz));
    const float qz = __builtin_fmaf(q0.z, dx, __builtin_fmaf(q1.x, dy, q1.y * dz));
    const float dqd = __builtin_fmaf(dx, qx, __builtin_fmaf(dy, qy, dz * qz));
    float s = __builtin_fmaf(b.w, inv3, inv5 * __builtin_fmaf(7.5f * inv2, dqd, -1.5f * q1.z));
    float t = -3.0f * inv5;
    s = __uint_as_float(__float_as_uint(s) & bits);
    t = __uint_as_float(__float_as_uint(t) & bits);
    r.x = __builtin_fmaf(dx, s, __builtin_fmaf(t, qx, r.x));
    r.y = __builtin_fmaf(dy, s, __builtin_fmaf(t, qy, r.y));
    r.z = __builtin_fmaf(dz, s, __builtin_fmaf(t, qz, r.z));
}

// The walk of one wave.  K: waves that share a group's sums; this one takes
// the classes k, k + K, ...
template <bool OCT, bool QUAD, bool SOFT, int STATS, int K>
struct FastWalk {
    static constexpr int kGroup = OCT ? 8 : 2;  // lanes a popped sibling group takes
    static constexpr int kPop = kWave / kGroup;
    static constexpr int kOwn = kClasses / K;
    static constexpr int kWide = wide_groups(OCT, QUAD);
    using Lds = WaveLds<OCT, QUAD>;
    using Node = std::conditional_t<OCT, OctRec, NodeRec>;
    static constexpr int kEnd = QUAD ? kMaskCap : kListCap;

    const WalkArgs &a;
    Lds &L;
    const Node *__restrict__ nodes;
    int k;                       // this wave among the group's K
    int lane, row, t;            // row and target of the summing phase
    float px, py, pz, eps2;
    int64_t base;                // first target
    int ntgt;                    // targets (1..16)
    uint32_t mask0;              // their mask
    float glo[3], ghi[3];        // their bounding box
    int sp = 0, mq = 0, lq = 0, nfull = 0, npart = 0;
    int sums = 0;                // lists summed since the last addition to FP64
    bool fail = false;
    uint32_t np = 0;
    uint64_t pp = 0;
    uint32_t visits = 0, vlanes = 0, lvisits = 0, llanes = 0;
    Pair3 r[kOwn];
    double s[kOwn][3];

    __device__ __forceinline__ FastWalk(const WalkArgs &args, Lds &lds) : a(args), L(lds) {
        if constexpr (OCT) nodes = args.onodes;
        else nodes = args.nodes;
#pragma unroll
        for (int j = 0; j < kOwn; ++j) {
            r[j] = Pair3{0.0f, 0.0f, 0.0f};
            s[j][0] = 0.0; s[j][1] = 0.0; s[j][2] = 0.0;
        }
    }

    __device__ __forceinline__ void to_f64() {
#pragma unroll
        for (int j = 0; j < kOwn; ++j) {
            s[j][0] += (double)r[j].x; s[j][1] += (double)r[j].y; s[j][2] += (double)r[j].z;
            r[j] = Pair3{0.0f, 0.0f, 0.0f};
        }
        sums = 0;
    }

    __device__ __forceinline__ uint32_t bits_of(uint16_t m) const {
        return (uint32_t)__builtin_amdgcn_sbfe((int32_t)m, (uint32_t)t, 1u);
    }

    // ---- summing: the last 64 entries of a list
    __device__ __forceinline__ void summed() {
        lds_order();
        if (++sums >= kFlushEvery) to_f64();
    }
    __device__ __forceinline__ void sum_full() {
        lds_order();
        nfull -= kWave;
        const float4 *p = L.src + nfull + row;
#pragma unroll
        for (int j = 0; j < kOwn; ++j)
#pragma unroll
            for (int i = 0; i < kSub / kRows; ++i)
                add_source<SOFT, false>(p[(k + j * K) * kSub + i * kRows], 0u, px, py, pz, eps2, r[j]);
        summed();
    }
    // Entries first .. first + 15 of the masked list.
    __device__ __forceinline__ void sum_chunk_part(int first, int j) {
#pragma unroll
        for (int i = 0; i < kSub / kRows; ++i) {
            const int e = first + i * kRows + row;
            add_source<SOFT, true>(L.src[kEnd - 1 - e], bits_of(L.smask[e]), px, py, pz, eps2, r[j]);
        }
    }
    __device__ __forceinline__ void sum_part() {
        lds_order();
        npart -= kWave;
#pragma unroll
        for (int j = 0; j < kOwn; ++j) sum_chunk_part(npart + (k + j * K) * kSub, j);
        summed();
    }
    __device__ __forceinline__ void sum_chunk_quad(int first, int j) {
        if constexpr (QUAD) {
#pragma unroll
            for (int i = 0; i < kSub / kRows; ++i) {
                const int e = first + i * kRows + row;
                add_quad<SOFT>(L.qsrc[0][e], L.qsrc[1][e], L.qsrc[2][e], bits_of(L.qmask[e]), px, py, pz, eps2, r[j]);
            }
        }
    }
    __device__ __forceinline__ void sum_quad() {
        lds_order();
        nfull -= kWave;
#pragma unroll
        for (int j = 0; j < kOwn; ++j) sum_chunk_quad(nfull + (k + j * K) * kSub, j);
        summed();
    }
    __device__ __forceinline__ void sum_ready() {
        if constexpr (QUAD) {
            if (nfull >= kWave) sum_quad();
        } else {
            if (nfull >= kWave) sum_full();
        }
        if (npart >= kWave) sum_part();
    }
    // What is left of the lists: entries 16 c .. 16 c + 15 are class c mod 4;
    // the last chunk is filled up with sources that no target takes.
    __device__ __forceinline__ void sum_rest() {
        lds_order();
        if constexpr (!QUAD) {
            // at most 63 + 63 entries: the moved ones stay clear of the others
            if (lane < nfull) {
                L.src[kEnd - 1 - npart - lane] = L.src[lane];
                L.smask[npart + lane] = (uint16_t)mask0;
            }
            npart += nfull;
            nfull = 0;
        } else {
            const int end = (nfull + kSub - 1) & ~(kSub - 1);
            if (lane < end - nfull) {
#pragma unroll
                for (int i = 0; i < 3; ++i) L.qsrc[i][nfull + lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                L.qmask[nfull + lane] = 0;
            }
            lds_order();
#pragma unroll
            for (int j = 0; j < kOwn; ++j)
                if ((k + j * K) * kSub < end) sum_chunk_quad((k + j * K) * kSub, j);
        }
        const int end = (npart + kSub - 1) & ~(kSub - 1);
        if (lane < end - npart) {
            L.src[kEnd - 1 - npart - lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            L.smask[npart + lane] = 0;
        }
        lds_order();
        for (int c0 = 0; c0 < 2 * kClasses; c0 += kClasses)
#pragma unroll
            for (int j = 0; j < kOwn; ++j) {
                const int c = c0 + k + j * K;
                if (c * kSub < end) sum_chunk_part(c * kSub, j);
            }
        to_f64();
    }

    // ---- listing
    // Source b for the targets in m (lanes in pred; bodies and monopole nodes).
    __device__ __forceinline__ void list_source(uint64_t pred, float4 b, uint32_t m) {
        uint64_t g = pred;
        if constexpr (!QUAD) {
            const uint64_t all = __ballot(m == mask0), f = pred & all;
            g = pred & ~all;
            if (in_lane(f)) L.src[nfull + rank_in(f)] = b;
            nfull += __popcll(f);
        }
        if (in_lane(g)) {
            const int e = npart + rank_in(g);
            L.src[kEnd - 1 - e] = b;
            L.smask[e] = (uint16_t)m;
        }
        npart += __popcll(g);
    }
    // Node `node`, accepted by the targets in m.
    __device__ __forceinline__ void list_node(uint64_t pred, int node, float4 com, uint32_t m) {
        if (STATS >= 1 && in_lane(pred)) np += __popc(m);
        if constexpr (QUAD) {
            if (in_lane(pred)) {
                const int e = nfull + rank_in(pred);
                L.qsrc[0][e] = com;
                L.qsrc[1][e] = a.quad[2 * (int64_t)node];
                L.qsrc[2][e] = a.quad[2 * (int64_t)node + 1];
                L.qmask[e] = (uint16_t)m;
            }
            nfull += __popcll(pred);
        } else {
            list_source(pred, com, m);
        }
    }
    // A node opened by the targets in m: its children to the stack, or its
    // bodies' range to the leaf queue.
    __device__ __forceinline__ void open_node(uint64_t pred, int4 topo, int nch, uint32_t m) {
        const uint64_t inner = __ballot(topo.z >= 0), bi = pred & inner, bl = pred & ~inner;
        const int ni = __popcll(bi), nl = __popcll(bl);
        if (sp + ni > Lds::kStack || lq + nl > kLeafCap) {  // unreachable
            fail = true;
            return;
        }
        if (in_lane(bi)) {
            const int e = sp + rank_in(bi);
            L.st_node[e] = OCT ? topo.z | ((nch - 1) << 28) : topo.z;
            L.st_mask[e] = (uint16_t)m;
        }
        if (in_lane(bl)) {
            const int e = lq + rank_in(bl);
            const bool ok = (uint32_t)topo.x < (uint32_t)a.n && (uint32_t)topo.y <= (uint32_t)a.n - (uint32_t)topo.x;
            if (!ok) fail = true;
            L.lq_first[e] = ok ? topo.x : 0;
            L.lq_cnt[e] = ok ? topo.y : 0;
            L.lq_mask[e] = (uint16_t)m;
            if (STATS >= 1 && ok) pp += (uint64_t)__popc(m) * (uint64_t)(uint32_t)topo.y;
            if (STATS >= 2) { lvisits += 1; llanes += __popc(m); }
        }
        sp += ni;
        lq += nl;
    }

    // The next 64 bodies of the queued leaves, from the last one on, one a lane:
    // a scan of the leaves' counts tells each lane its leaf, so that the lanes
    // are full whatever the leaves hold.  A pass over 1,024 systems of 256 to
    // 65,536 bodies, ms, at leaf size 16 / 32 / 64: linear BVH 38.7 / 53.2 /
    // 73.1, octree 24.5 / 26.4 / 33.3; four leaves of at most 16 bodies or one
    // larger leaf at a time took 40.9 / 87.0 / 94.7 and 26.5 / 34.3 / 43.6.
    // Leaves of 20 bodies or more summed by themselves, without the list and
    // its masks: 10 to 20 % slower (part-filled chunks cost more than masks).
    struct Bodies {
        float4 b;    // a lane's body
        uint32_t m;  // the targets that take it
        int n;       // lanes with a body
    };
    __device__ __forceinline__ Bodies next_bodies() {
        lds_order();
        // lane = queued leaf
        const int e = lq - 1 - lane;
        int first = 0, cnt = 0;
        uint32_t m = 0;
        if (e >= 0) {
            first = L.lq_first[e];
            cnt = L.lq_cnt[e];
            m = L.lq_mask[e];
        }
        // a leaf's bodies go to the lanes from excl on
        const int c = cnt < kWave + 1 ? cnt : kWave + 1;
        const int incl = incl_scan(c), excl = incl - c;
        if (lane < 2) L.starts[lane] = 0;
        lds_order();
        if (c > 0 && excl < kWave) atomicOr(&L.starts[excl >> 5], 1u << (excl & 31));
        const int done = __popcll(__ballot(e >= 0 && incl <= kWave));
        if (e >= 0 && excl < kWave && incl > kWave) {  // the rest of this leaf waits
            L.lq_first[e] = first + (kWave - excl);
            L.lq_cnt[e] = cnt - (kWave - excl);
        }
        lq -= done;
        lds_order();
        const uint64_t starts = uniform_u64((uint64_t)L.starts[1] << 32 | L.starts[0]);
        const int from = 4 * rank_in(starts >> 1);  // lane of this lane's leaf, in bytes
        const int at = __builtin_amdgcn_ds_bpermute(from, first - excl) + lane;
        Bodies r;
        r.m = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)m);
        const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
        r.n = total < kWave ? total : kWave;
        r.b = a.bodies[lane < r.n ? at : 0];
        return r;
    }
    __device__ __forceinline__ void list_bodies(const Bodies &v) {
        list_source(lanes_below(v.n), v.b, v.m);
        sum_ready();
    }
    // Lists bodies of the queued leaves while more than `keep` leaves wait; the
    // next ones are on their way while the present ones are listed and summed.
    __device__ __forceinline__ void expand_leaves(int keep) {
        if (lq <= keep) return;
        Bodies now = next_bodies();
        while (lq > keep) {
            const Bodies then = next_bodies();
            list_bodies(now);
            now = then;
        }
        list_bodies(now);
    }

    // The criterion against the targets' box: the lanes whose node every point
    // of it accepts / rejects.
    __device__ __forceinline__ void box_test(const Node &nd, uint64_t &acc, uint64_t &rej) const {
        float c[3], thr;
        if constexpr (OCT) { c[0] = nd.com.x; c[1] = nd.com.y; c[2] = nd.com.z; thr = nd.lo.w; }
        else { c[0] = nd.mac.x; c[1] = nd.mac.y; c[2] = nd.mac.z; thr = nd.mac.w; }
        float lo2[3], hi2[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float u = glo[d] - c[d], v = c[d] - ghi[d];
            const float near = fmaxf(fmaxf(u, v), 0.0f), far = fmaxf(fabsf(u), fabsf(v));
            lo2[d] = near * near;
            hi2[d] = far * far;
        }
        acc = __ballot((lo2[0] + lo2[1]) + lo2[2] > thr);
        rej = ~__ballot((hi2[0] + hi2[1]) + hi2[2] > thr);
        if constexpr (OCT) {
            // the exclusion region [lo, hi) around the cell
            acc &= __ballot(ghi[0] < nd.lo.x) | __ballot(ghi[1] < nd.lo.y) | __ballot(ghi[2] < nd.lo.z) |
                   __ballot(glo[0] >= nd.hi.x) | __ballot(glo[1] >= nd.hi.y) | __ballot(glo[2] >= nd.hi.z);
            rej |= __ballot(glo[0] >= nd.lo.x) & __ballot(glo[1] >= nd.lo.y) & __ballot(glo[2] >= nd.lo.z) &
                   __ballot(ghi[0] < nd.hi.x) & __ballot(ghi[1] < nd.hi.y) & __ballot(ghi[2] < nd.hi.z);
        }
    }

    __device__ __forceinline__ static int children_of(const Node &nd) {
        if constexpr (OCT) return oct_nchild(nd);
        else return 2;
    }

    // Pops sibling groups, one node per lane, and tests them against the box.
    __device__ __forceinline__ void step() {
        int p = sp < kPop ? sp : kPop;
        const int room = (kWide - sp) / (kGroup - 1);
        if (p > room) p = room > 1 ? room : 1;
        sp -= p;
        lds_order();
        const int e = lane / kGroup, c = lane % kGroup;
        bool ok = e < p;
        int node = 0;
        uint32_t m = 0;
        if (ok) {
            const int enc = L.st_node[sp + e];
            m = L.st_mask[sp + e];
            if constexpr (OCT) {
                node = (enc & 0x0FFFFFFF) + c;
                ok = c <= (int)((uint32_t)enc >> 28);
            } else {
                node = (enc & 0x3FFFFFFF) + c;
                ok = c == 0 || !(enc & 0x40000000);  // the root has no sibling
            }
        }
        lds_order();
        if (ok && (uint32_t)node >= (uint32_t)a.max_nodes) { fail = true; ok = false; }
        const uint64_t okm = __ballot(ok);
        const Node nd = nodes[ok ? node : 0];
        uint64_t acc, rej;
        box_test(nd, acc, rej);
        acc &= okm;
        rej &= okm & ~acc;
        if (STATS >= 2 && ok) { visits += 1; vlanes += __popc(m); }
        const uint64_t mix = okm & ~acc & ~rej;
        if (in_lane(mix)) {
            const int x = mq + rank_in(mix);
            L.mq_node[x] = node;
            L.mq_mask[x] = (uint16_t)m;
        }
        mq += __popcll(mix);
        list_node(acc, node, nd.com, m);
        open_node(rej, nd.topo, children_of(nd), m);
    }

    // Up to 64 nodes on which the targets differ, each against every target.
    __device__ __forceinline__ void mixed() {
        const int room = kWide - sp;
        int p = mq < kWave ? mq : kWave;
        if (p > room) p = room > 1 ? room : 1;
        mq -= p;
        lds_order();
        const bool ok = lane < p;
        int node = 0;
        uint32_t m = 0;
        if (ok) {
            node = L.mq_node[mq + lane];
            m = L.mq_mask[mq + lane];
        }
        lds_order();
        const Node nd = nodes[node];  // checked when it was queued (0 in the lanes past p)
        const const_ptr<Body4> tg = as_const(reinterpret_cast<const Body4 *>(a.targets + base));
        uint32_t acc = 0;  // bit i: target i accepts
#pragma unroll
        for (int i = kSub - 1; i >= 0; --i) {
            uint64_t hit = 0;
            if (i < ntgt) {
                const Body4 q = load_body(tg + i);
                if constexpr (OCT) {
                    const float dx = q.x - nd.com.x, dy = q.y - nd.com.y, dz = q.z - nd.com.z;
                    hit = __ballot(dx * dx + dy * dy + dz * dz > nd.lo.w) &
                          ~(__ballot(nd.lo.x <= q.x) & __ballot(nd.lo.y <= q.y) & __ballot(nd.lo.z <= q.z) &
                            __ballot(q.x < nd.hi.x) & __ballot(q.y < nd.hi.y) & __ballot(q.z < nd.hi.z));
                } else {
                    const float dx = q.x - nd.mac.x, dy = q.y - nd.mac.y, dz = q.z - nd.mac.z;
                    hit = __ballot(dx * dx + dy * dy + dz * dz > nd.mac.w);
                }
            }
            acc = shift_in(acc, hit);
        }
        const uint32_t take = acc & m, open = m & ~acc;
        list_node(__ballot(take != 0), node, nd.com, take);
        open_node(__ballot(open != 0), nd.topo, children_of(nd), open);
    }

    __device__ __forceinline__ void walk(int root) {
        if (lane == 0) {
            L.st_node[0] = OCT ? root : root | 0x40000000;
            L.st_mask[0] = (uint16_t)mask0;
        }
        sp = 1;
        uint32_t iters = 0;
        while (sp > 0 || mq > 0) {
            if (__builtin_expect(++iters > kMaxFastIters, 0)) { fail = true; break; }
            if (mq >= kWave || sp == 0 || (mq > 0 && sp >= kWide)) mixed();
            else step();
            if (__ballot(fail)) break;
            sum_ready();
            expand_leaves(sp > 0 || mq > 0 ? kLeafKeep : 0);
        }
        if (__ballot(fail)) return;  // the lists may hold more than a walk that went on would leave in them
        sum_rest();
    }
};

// FAST walk kernel.  FOREST: the wave's system from the forest's wave table
// (wave_task).  K waves serve each 16 targets (1, 2 or 4).
template <bool OCT, bool QUAD, bool SOFT, int STATS, bool FOREST, int K>
__device__ __forceinline__ void walk_fast(const WalkArgs &a, WaveLds<OCT, QUAD> *lds, double (*cls)[kClasses][3][kSub]) {
    const int lane = lane_id();
    const int wv = uniform_i32(threadIdx.x / kWave);
    const int64_t gw = (int64_t)walk_block<FOREST>() * kFastWaves + wv;
    const int64_t sub = gw / K;
    const int k = (int)(gw - sub * K);
    const WaveTask T = wave_task<FOREST>(a, sub / kRows);
    const int64_t base = T.base + (sub % kRows) * kSub;
    const bool any = base < T.end;
    bool root_ok = true;
    if (FOREST) root_ok = T.root >= 0 && T.root < a.max_nodes;

    FastWalk<OCT, QUAD, SOFT, STATS, K> w(a, lds[wv]);
    w.k = k;
    w.lane = lane;
    w.row = lane / kSub;
    w.t = lane % kSub;
    w.base = base;
    w.eps2 = T.eps2;
    w.px = 0.0f; w.py = 0.0f; w.pz = 0.0f;
    w.ntgt = any ? (int)(T.end - base < kSub ? T.end - base : kSub) : 0;
    w.mask0 = (1u << w.ntgt) - 1u;
    if (any && root_ok) {
        // lanes past the last target repeat it: the box is that of the targets
        const float4 me = a.targets[base + (w.t < w.ntgt ? w.t : w.ntgt - 1)];
        w.px = me.x; w.py = me.y; w.pz = me.z;
        float lo[3] = {me.x, me.y, me.z}, hi[3] = {me.x, me.y, me.z};
#pragma unroll
        for (int o = kSub / 2; o > 0; o >>= 1)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, kWave));
                hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, kWave));
            }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            w.glo[d] = readlane_f32(lo[d], 0);
            w.ghi[d] = readlane_f32(hi[d], 0);
        }
        w.walk(T.root);
    }
    if (any && !root_ok) w.fail = true;
    if (__ballot(w.fail) && lane == 0) atomicOr(a.err, 2u);

    // the rows' sums, then the classes'
    double tot[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        double c[w.kOwn];
#pragma unroll
        for (int j = 0; j < w.kOwn; ++j) {
            c[j] = w.s[j][d];
            c[j] += __shfl_xor(c[j], kSub, kWave);
            c[j] += __shfl_xor(c[j], 2 * kSub, kWave);
        }
        if constexpr (K == 1) {
            tot[d] = (c[0] + c[1]) + (c[2] + c[3]);
        } else if (lane < kSub) {
#pragma unroll
            for (int j = 0; j < w.kOwn; ++j) cls[wv / K][k + j * K][d][lane] = c[j];
        }
    }
    if constexpr (K > 1) {
        __syncthreads();
        if (k == 0 && lane < kSub) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const auto &g = cls[wv / K];
                tot[d] = (g[0][d][lane] + g[1][d][lane]) + (g[2][d][lane] + g[3][d][lane]);
            }
        }
    }
    if (k != 0) return;
    if (lane < w.ntgt) {
        const uint32_t o = a.perm[base + lane];
        if ((int64_t)o < a.nt) {
            const double g = (double)T.G;
            a.ax[o] = (float)(tot[0] * g);
            a.ay[o] = (float)(tot[1] * g);
            a.az[o] = (float)(tot[2] * g);
        }
    }
    if (STATS >= 1) {
        auto total = [](uint64_t v) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor((unsigned long long)v, o, kWave);
            return (unsigned long long)v;
        };
        const unsigned long long pp = total(w.pp), np = total(w.np);
        if (lane == 0) {
            atomicAdd(&a.counts[0], pp);
            atomicAdd(&a.counts[1], np);
        }
        if (STATS >= 2) {
            const unsigned long long v = total(w.visits), vl = total(w.vlanes), l = total(w.lvisits), ll = total(w.llanes);
            if (lane == 0) {
                atomicAdd(&a.counts[2], v);
                atomicAdd(&a.counts[3], vl);
                atomicAdd(&a.counts[4], l);
                atomicAdd(&a.counts[5], ll);
            }
        }
    }
}

template <bool QUAD, bool SOFT, int STATS, bool FOREST, int K>
__global__ __launch_bounds__(64 * kFastWaves) void k_walk_lbvh_fast(WalkArgs a) {
    __shared__ WaveLds<false, QUAD> lds[kFastWaves];
    __shared__ double cls[K > 1 ? kFastWaves / K : 1][kClasses][3][kSub];
    walk_fast<false, QUAD, SOFT, STATS, FOREST, K>(a, lds, cls);
}

template <bool QUAD, bool SOFT, int STATS, bool FOREST, int K>
__global__ __launch_bounds__(64 * kFastWaves) void k_walk_oct_fast(WalkArgs a) {
    __shared__ WaveLds<true, QUAD> lds[kFastWaves];
    __shared__ double cls[K > 1 ? kFastWaves / K : 1][kClasses][3][kSub];
    walk_fast<true, QUAD, SOFT, STATS, FOREST, K>(a, lds, cls);
}

template <bool OCT, bool QUAD, bool SOFT, int STATS, bool FOREST, int K>
static void launch_k(const WalkArgs &a, int64_t groups, hipStream_t s) {
    const dim3 g((unsigned)(groups * K)), t(64 * kFastWaves);
    if constexpr (OCT) hipLaunchKernelGGL((k_walk_oct_fast<QUAD, SOFT, STATS, FOREST, K>), g, t, 0, s, a);
    else hipLaunchKernelGGL((k_walk_lbvh_fast<QUAD, SOFT, STATS, FOREST, K>), g, t, 0, s, a);
}

template <bool OCT, bool QUAD, bool SOFT, int STATS>
static void launch_s(const WalkArgs &a, hipStream_t s) {
    static_assert(kFastWaves == kRows, "a workgroup's waves serve 64 targets (over K)");
    const int64_t groups = a.nsys > 0 ? a.nwaves : (a.nt + kWave - 1) / kWave;
    if (a.nsys > 0) {
        if (a.split >= 4) launch_k<OCT, QUAD, SOFT, STATS, true, 4>(a, groups, s);
        else if (a.split >= 2) launch_k<OCT, QUAD, SOFT, STATS, true, 2>(a, groups, s);
        else launch_k<OCT, QUAD, SOFT, STATS, true, 1>(a, groups, s);
    } else {
        if (a.split >= 4) launch_k<OCT, QUAD, SOFT, STATS, false, 4>(a, groups, s);
        else if (a.split >= 2) launch_k<OCT, QUAD, SOFT, STATS, false, 2>(a, groups, s);
        else launch_k<OCT, QUAD, SOFT, STATS, false, 1>(a, groups, s);
    }
}

template <bool OCT, int STATS>
static void launch_q(const WalkArgs &a, hipStream_t s) {
    if (a.quad) {
        if (a.eps2 > 0.0f) launch_s<OCT, true, true, STATS>(a, s);
        else launch_s<OCT, true, false, STATS>(a, s);
    } else {
        if (a.eps2 > 0.0f) launch_s<OCT, false, true, STATS>(a, s);
        else launch_s<OCT, false, false, STATS>(a, s);
    }
}

void launch_walk_fast(const WalkArgs &a, bool octree, int stats, hipStream_t s) {
    if (octree) {
        if (stats >= 2) launch_q<true, 2>(a, s);
        else if (stats == 1) launch_q<true, 1>(a, s);
        else launch_q<true, 0>(a, s);
    } else {
        if (stats >= 2) launch_q<false, 2>(a, s);
        else if (stats == 1) launch_q<false, 1>(a, s);
        else launch_q<false, 0>(a, s);
    }
}

}  // namespace nbg
