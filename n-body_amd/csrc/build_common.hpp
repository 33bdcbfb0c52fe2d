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

// The kernels that compute the keys take few workgroups, since each adds its
// digit counts to the sort's histograms, and more threads in each where a
// thread would have many bodies.  Keys phase, us, 256 workgroups of 256
// threads at every size / this rule: octree paths, 1,000,000 bodies 56 / 36,
// 4,000,000 199 / 92, 16,777,216 832 / 331; 63-bit codes 21 / 18, 54 / 33, 239 /
// 90.  1,024 threads for 70,000 bodies 16 to 14, 512 workgroups for 1,000,000
// codes 22 to 18, for 16,777,216 90 to 105.
constexpr int kKeyThreads = 1024;
inline int key_threads(int64_t n) { return n <= 131072 ? 256 : kKeyThreads; }
inline unsigned key_blocks(int64_t n) {
    const int64_t g = (n + key_threads(n) - 1) / key_threads(n), most = n < ((int64_t)1 << 22) ? 256 : 512;
    return (unsigned)(g < most ? g : most);
}

// Second stage, at the start of the kernel that computes the keys: every
// workgroup folds the per-block partials (the kernel boundary makes them
// visible; no agent-scope fence, which on gfx950 is an L2 write-back +
// invalidate) into bb, in one order, and the first one stores the box.
__device__ __forceinline__ void fold_bbox(const float *__restrict__ partials, int blocks, float *bb, float *out6) {
    __shared__ float s_part[kKeyThreads / kWave][6];
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int b = threadIdx.x; b < blocks; b += blockDim.x)
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
    for (int ww = 1; ww < (int)blockDim.x / kWave; ++ww)
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
