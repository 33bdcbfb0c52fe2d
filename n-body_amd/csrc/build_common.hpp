// Device helpers of both tree builds (build.hip, octree.hip).
#pragma once

#include <cfloat>

#include "device.hpp"
#include "launch.hpp"

namespace nbg {

// glm::min(x, y) = (y < x) ? y : x and glm::max(x, y) = (x < y) ? y : x; the
// argument order matters only for ties between +0 and -0.
__device__ __forceinline__ float fmin_ref(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float fmax_ref(float a, float b) { return (a < b) ? b : a; }

// Second stage, at the start of the kernel that computes the keys: every
// workgroup folds the per-block partials (the kernel boundary makes them
// visible; no agent-scope fence, which on gfx950 is an L2 write-back +
// invalidate) into bb, in one order, and the first one stores the box.
__device__ __forceinline__ void fold_bbox(const float *__restrict__ partials, int blocks, float *bb, float *out6) {
    __shared__ float s_part[4][6];
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int b = threadIdx.x; b < blocks; b += 256)
        for (int d = 0; d < 3; ++d) {
            mn[d] = fmin_ref(mn[d], partials[b * 6 + d]);
            mx[d] = fmax_ref(mx[d], partials[b * 6 + 3 + d]);
        }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            mn[d] = fmin_ref(mn[d], __shfl_xor(mn[d], o, kWave));
            mx[d] = fmax_ref(mx[d], __shfl_xor(mx[d], o, kWave));
        }
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0)
        for (int d = 0; d < 3; ++d) { s_part[w][d] = mn[d]; s_part[w][3 + d] = mx[d]; }
    __syncthreads();
    for (int d = 0; d < 3; ++d) { mn[d] = s_part[0][d]; mx[d] = s_part[0][3 + d]; }
    for (int ww = 1; ww < 4; ++ww)
        for (int d = 0; d < 3; ++d) { mn[d] = fmin_ref(mn[d], s_part[ww][d]); mx[d] = fmax_ref(mx[d], s_part[ww][3 + d]); }
    for (int d = 0; d < 3; ++d) { bb[d] = mn[d]; bb[3 + d] = mx[d]; }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        for (int d = 0; d < 6; ++d) out6[d] = bb[d];
}

// Digit counts of a workgroup's keys in LDS, added to the sort's histograms.
struct DigitCount {
    uint32_t *h;
    int passes, shift;
    __device__ __forceinline__ void clear() const {
        for (int i = threadIdx.x; i < passes * kRadix; i += blockDim.x) h[i] = 0;
    }
    template <typename K>
    __device__ __forceinline__ void add(K k) const {
        for (int p = 0; p < passes; ++p) atomicAdd(&h[p * kRadix + (uint32_t)((k >> (shift + 8 * p)) & 0xFF)], 1u);
    }
    __device__ __forceinline__ void store(uint32_t *ghist) const {
        for (int i = threadIdx.x; i < passes * kRadix; i += blockDim.x) {
            const uint32_t v = h[i];
            if (v) atomicAdd(&ghist[i], v);
        }
    }
};

// Adds item i's value to its scan tile's sum (cleared; one atomic a wave;
// sums null: the scan adds them up itself).
// The active lanes are a wave's first ones and share a tile (tiles are
// multiples of a wave), so lane 0 gathers them all.
__device__ __forceinline__ void scan_sum(uint32_t v, int64_t i, uint32_t *sums) {
    if (!sums) return;
    const int active = __popcll(__ballot(true)), l = lane_id();
    uint32_t t = v;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t u = __shfl_down(t, o, kWave);
        t += l + o < active ? u : 0u;
    }
    if (l == 0 && t) atomicAdd(&sums[i / kScanTile], t);
}

}  // namespace nbg
