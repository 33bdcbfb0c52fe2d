// The order in which a walk takes its targets, for gfx950.
//
// A walk's waves take 16 (or 64) consecutive targets, and its work grows with
// the size of their box: runs of the Morton order straddle cells.  Here every
// kGroupBlock consecutive bodies of the Morton order are split at the median
// of the longest side of their box, again and again down to 16, so that each
// 16 consecutive targets (and 32, 64, ...) fill a compact box.  On a model of
// the walk (200,000 and 1,000,000 Plummer bodies, theta 0.5) that takes 8.3 to
// 8.7 % off its instructions, 256 bodies a block 7.4 %, a Hilbert order 6.5 %,
// one block for all 10 %.  Measured, FAST walk of 1,048,576 bodies: linear BVH
// 5.16 -> 4.60 ms, octree 2.04 -> 1.86, quadrupole linear BVH of 500,000 1.88
// -> 1.66.
//
// A workgroup sorts a block in registers, 4 consecutive slots a lane: six
// bitonic sorts, of segments of 1,024 down to 32, by the coordinate along the
// segment's longest side (22 bits of it, and the body's number: keys differ,
// so the order is a function of the block alone).  84 of the 200 steps stay
// within a lane, one instruction a slot, 112 exchange lanes in the vector
// unit, 4 cross waves.  30 us for 1,048,576 bodies and 15 for 20,000 (with 16
// slots a lane and a wave a block 49 and 35, with one slot a lane 70 and 20):
// vector issue, then the steps' latency.

#include "device.hpp"
#include "launch.hpp"

#include <type_traits>

namespace nbg {

constexpr int kGroupBlock = 1024;
constexpr int kSlots = 4;  // of a lane, consecutive
constexpr int kGroupThreads = kGroupBlock / kSlots;
using SlotKeys = uint32_t[kSlots][kGroupThreads];
using Boxes = float[kGroupThreads / kWave][6];

// v of lane ^ X.
template <int X>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    constexpr int kQuad = 0x1B, kHalfMirror = 0x141, kMirror = 0x140, kRor8 = 0x128;
    auto dpp = [](uint32_t u, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_mov_dpp((int)u, decltype(ctrl)::value, 0xF, 0xF, true);
    };
    constexpr int R = X & 15;  // within a row of 16
    static_assert(R == 0 || R == 1 || R == 2 || R == 3 || R == 4 || R == 7 || R == 8 || R == 15, "no permute for it");
    if constexpr (R == 1) v = dpp(v, std::integral_constant<int, 0xB1>{});  // quad_perm 1 0 3 2
    if constexpr (R == 2) v = dpp(v, std::integral_constant<int, 0x4E>{});  // quad_perm 2 3 0 1
    if constexpr (R == 3) v = dpp(v, std::integral_constant<int, kQuad>{});  // quad_perm 3 2 1 0
    if constexpr (R == 4) v = dpp(dpp(v, std::integral_constant<int, kHalfMirror>{}), std::integral_constant<int, kQuad>{});
    if constexpr (R == 7) v = dpp(v, std::integral_constant<int, kHalfMirror>{});
    if constexpr (R == 8) v = dpp(v, std::integral_constant<int, kRor8>{});
    if constexpr (R == 15) v = dpp(v, std::integral_constant<int, kMirror>{});
    if constexpr (X & 16) {
        const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        v = lane_id() & 16 ? p[0] : p[1];
    }
    if constexpr (X & 32) {
        const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        v = lane_id() & 32 ? p[0] : p[1];
    }
    return v;
}

// Slot e of this lane and slot e ^ J, J < kSlots: the smaller to the lower one.
template <int J>
__device__ __forceinline__ void step_in_lane(uint32_t (&v)[kSlots]) {
#pragma unroll
    for (int e = 0; e < kSlots; ++e) {
        if ((e ^ J) < e) continue;
        const uint32_t a = v[e], b = v[e ^ J];
        v[e] = a < b ? a : b;
        v[e ^ J] = a < b ? b : a;
    }
}
// Slot e of this thread and slot e (MIRROR: the mirrored slot) of thread ^ X.
template <int X, bool MIRROR>
__device__ __forceinline__ void step_lanes(uint32_t (&v)[kSlots], SlotKeys &s_key) {
    constexpr int kTop = MIRROR ? (X + 1) / 2 : X;  // the highest bit of X
    const bool low = (threadIdx.x & kTop) == 0;
    uint32_t o[kSlots];
    if constexpr (X >= kWave) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kSlots; ++e) s_key[e][threadIdx.x] = v[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kSlots; ++e) o[e] = s_key[MIRROR ? kSlots - 1 - e : e][threadIdx.x ^ X];
    } else {
#pragma unroll
        for (int e = 0; e < kSlots; ++e) o[e] = lane_xor<X>(v[MIRROR ? kSlots - 1 - e : e]);
    }
#pragma unroll
    for (int e = 0; e < kSlots; ++e) v[e] = (v[e] < o[e]) == low ? v[e] : o[e];
}
template <int J>
__device__ __forceinline__ void merge_from(uint32_t (&v)[kSlots], SlotKeys &s_key) {
    if constexpr (J >= kSlots) step_lanes<J / kSlots, false>(v, s_key);
    else if constexpr (J >= 1) step_in_lane<J>(v);
    if constexpr (J > 1) merge_from<J / 2>(v, s_key);
}
// Sorts segments of S slots: merges of sorted halves, the first step of each
// against the mirrored slot, so that every merge ascends.
template <int S, int K = 2>
__device__ __forceinline__ void sort_segments(uint32_t (&v)[kSlots], SlotKeys &s_key) {
    if constexpr (K <= kSlots) step_in_lane<K - 1>(v);
    else step_lanes<K / kSlots - 1, true>(v, s_key);
    merge_from<K / 4>(v, s_key);
    if constexpr (K < S) sort_segments<S, 2 * K>(v, s_key);
}

template <int X>
__device__ __forceinline__ void box_step(float (&lo)[3], float (&hi)[3]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        lo[d] = fminf(lo[d], __uint_as_float(lane_xor<X>(__float_as_uint(lo[d]))));
        hi[d] = fmaxf(hi[d], __uint_as_float(lane_xor<X>(__float_as_uint(hi[d]))));
    }
}

// Splits the segments of S slots; v: the slots' bodies (numbers in the block),
// in the low 10 bits, in and out.  Numbers from cnt on are empty and stay last.
template <int S>
__device__ __forceinline__ void split_segments(uint32_t (&v)[kSlots], int cnt, const float (&s_pos)[3][kGroupBlock],
                                               Boxes &s_box, SlotKeys &s_key) {
    float lo[3], hi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) { lo[d] = __builtin_huge_valf(); hi[d] = -__builtin_huge_valf(); }
#pragma unroll
    for (int e = 0; e < kSlots; ++e) {
        const int body = v[e] & (kGroupBlock - 1);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float c = s_pos[d][body];
            lo[d] = fminf(lo[d], body < cnt ? c : lo[d]);
            hi[d] = fmaxf(hi[d], body < cnt ? c : hi[d]);
        }
    }
    box_step<1>(lo, hi);
    if constexpr (S > 2 * kSlots) box_step<2>(lo, hi);
    if constexpr (S > 4 * kSlots) box_step<4>(lo, hi);
    if constexpr (S > 8 * kSlots) box_step<8>(lo, hi);
    if constexpr (S > 16 * kSlots) box_step<16>(lo, hi);
    if constexpr (S > 32 * kSlots) box_step<32>(lo, hi);
    if constexpr (S > kWave * kSlots) {
        constexpr int W = S / (kWave * kSlots);  // waves of a segment
        const int w = threadIdx.x / kWave;
        __syncthreads();
        if (lane_id() == 0)
            for (int d = 0; d < 3; ++d) { s_box[w][d] = lo[d]; s_box[w][3 + d] = hi[d]; }
        __syncthreads();
        for (int i = 0; i < W; ++i)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                lo[d] = fminf(lo[d], s_box[(w & ~(W - 1)) + i][d]);
                hi[d] = fmaxf(hi[d], s_box[(w & ~(W - 1)) + i][3 + d]);
            }
    }
    const float ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
    const bool use_y = ey > ex, use_z = ez > (use_y ? ey : ex);
    const int axis = use_z ? 2 : use_y ? 1 : 0;
    const float ext = use_z ? ez : use_y ? ey : ex, from = use_z ? lo[2] : use_y ? lo[1] : lo[0];
    // 22 bits; a box without extent, or not finite, leaves the order to the numbers
    constexpr float kTop = 4194302.0f;
    const float scale = kTop / ext;
    const float *pos = &s_pos[0][0] + axis * kGroupBlock;
#pragma unroll
    for (int e = 0; e < kSlots; ++e) {
        const int body = v[e] & (kGroupBlock - 1);
        const float q = fminf(fmaxf((pos[body] - from) * scale, 0.0f), kTop);
        v[e] = ((body < cnt ? (uint32_t)q : 0x3FFFFFu) << 10) | (uint32_t)body;
    }
    sort_segments<S>(v, s_key);
}

// FOREST: the blocks of system i are those from sys_first[i] / 1024 + i on, of
// which some stay empty; systems below kGroupMin keep their order.
template <bool FOREST>
__global__ __launch_bounds__(kGroupThreads) void k_group_targets(const float4 *__restrict__ bodies,
                                                         const uint32_t *__restrict__ perm, int64_t n,
                                                         const int64_t *__restrict__ sys_first, int nsys,
                                                         float4 *__restrict__ out, uint32_t *__restrict__ out_perm) {
    __shared__ float s_pos[3][kGroupBlock];
    __shared__ SlotKeys s_key;
    __shared__ Boxes s_box;
    int64_t first = 0, end = n, block = blockIdx.x;
    if (FOREST) {
        int lo = 0, hi = nsys;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (sys_first[mid] / kGroupBlock + mid <= block) lo = mid;
            else hi = mid;
        }
        first = sys_first[lo];
        end = sys_first[lo + 1];
        block -= first / kGroupBlock + lo;
    }
    const int64_t base = first + block * kGroupBlock;
    if (base >= end) return;  // the whole workgroup
    const int cnt = (int)(end - base < kGroupBlock ? end - base : kGroupBlock);
    const bool grouped = !FOREST || end - first >= kGroupMin;
    const int t = threadIdx.x;
    uint32_t v[kSlots];
    if (grouped) {
#pragma unroll
        for (int e = 0; e < kSlots; ++e) {
            const int i = e * kGroupThreads + t;
            const float4 b = bodies[base + (i < cnt ? i : cnt - 1)];
            s_pos[0][i] = b.x;
            s_pos[1][i] = b.y;
            s_pos[2][i] = b.z;
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kSlots; ++e) v[e] = (uint32_t)(t * kSlots + e);
        split_segments<1024>(v, cnt, s_pos, s_box, s_key);
        split_segments<512>(v, cnt, s_pos, s_box, s_key);
        split_segments<256>(v, cnt, s_pos, s_box, s_key);
        split_segments<128>(v, cnt, s_pos, s_box, s_key);
        split_segments<64>(v, cnt, s_pos, s_box, s_key);
        split_segments<32>(v, cnt, s_pos, s_box, s_key);
        uint32_t *const order = &s_key[0][0];
        __syncthreads();  // a wave may still read what the last exchange across waves (512 slots) left in s_key
#pragma unroll
        for (int e = 0; e < kSlots; ++e) order[t * kSlots + e] = v[e] & (kGroupBlock - 1);
        __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < kSlots; ++e) {
        const int i = e * kGroupThreads + t;
        if (i >= cnt) break;
        const int body = grouped ? (int)(&s_key[0][0])[i] : i;
        out[base + i] = bodies[base + body];
        out_perm[base + i] = perm[base + body];
    }
}

void launch_group_targets(const float4 *bodies, const uint32_t *perm, int64_t n, float4 *out, uint32_t *out_perm,
                          hipStream_t s) {
    const dim3 g((unsigned)((n + kGroupBlock - 1) / kGroupBlock));
    hipLaunchKernelGGL(k_group_targets<false>, g, dim3(kGroupThreads), 0, s, bodies, perm, n, nullptr, 1, out, out_perm);
}

void launch_group_targets_forest(const float4 *bodies, const uint32_t *perm, int64_t n, const int64_t *sys_first,
                                 int nsys, float4 *out, uint32_t *out_perm, hipStream_t s) {
    const dim3 g((unsigned)(n / kGroupBlock + nsys));
    hipLaunchKernelGGL(k_group_targets<true>, g, dim3(kGroupThreads), 0, s, bodies, perm, n, sys_first, nsys, out,
                       out_perm);
}

}  // namespace nbg
