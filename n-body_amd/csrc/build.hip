// Tree build kernels for gfx950: bounding box, Morton keys, onesweep radix
// sort, gather, Karras LBVH topology and atomic-flag bottom-up summaries.
//
// Arithmetic that feeds a tree decision is IEEE binary32 in the reference's
// operation order (this file is compiled with -ffp-contract=off), so keys,
// topology and summaries are bit-exact with the reference's CPU path.

#include <cfloat>

#include "build_common.hpp"
#include "device.hpp"
#include "launch.hpp"

namespace nbg {

// ------------------------------------------------------------------ fill
__global__ void k_fill_u32(uint32_t *p, uint32_t v, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__device__ __forceinline__ void set_ranges(const FillRanges &fills) {
    for (int f = 0; f < fills.k; ++f) {
        uint32_t *q = fills.r[f].p;
        const uint32_t v = fills.r[f].v;
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < fills.r[f].n;
             i += (int64_t)gridDim.x * blockDim.x)
            q[i] = v;
    }
}

void launch_fill_u32(uint32_t *p, uint32_t v, int64_t n, hipStream_t s) {
    if (n <= 0) return;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
}

__global__ __launch_bounds__(256) void k_fills(FillRanges fills) { set_ranges(fills); }

static void launch_more(const FillSet &f, hipStream_t s) {
    for (const FillRanges::Range &q : f.more) launch_fill_u32(q.p, q.v, q.n, s);
}

void launch_fills(const FillSet &f, hipStream_t s) {
    launch_more(f, s);
    int64_t most = 1;
    for (int i = 0; i < f.k; ++i) most = f.r[i].n > most ? f.r[i].n : most;
    int64_t blocks = (most + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_fills, dim3((unsigned)blocks), dim3(256), 0, s, static_cast<const FillRanges &>(f));
}

// ------------------------------------------------------------------ bbox
// outerBoundingBox (Physics/Summaries/SummaryType.h:73-81).  Min/max are
// exact, so a tree-shaped reduction equals the reference's serial loop for
// finite inputs (up to which of +0/-0 survives a tie).  The kernel that
// computes the keys folds the per-block partials (fold_bbox).
// The build's first kernel: it also clears the words that the later ones
// count in (a launch of its own for each cost 4 us at small sizes).
__global__ __launch_bounds__(256) void k_bbox(const float *__restrict__ x, const float *__restrict__ y,
                                              const float *__restrict__ z, int64_t n, float *partials, FillRanges fills) {
    set_ranges(fills);
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        float v[3] = {x[i], y[i], z[i]};
#pragma unroll
        for (int d = 0; d < 3; ++d) { mn[d] = fmin_ref(mn[d], v[d]); mx[d] = fmax_ref(mx[d], v[d]); }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            mn[d] = fmin_ref(mn[d], __shfl_xor(mn[d], o, kWave));
            mx[d] = fmax_ref(mx[d], __shfl_xor(mx[d], o, kWave));
        }
    __shared__ float s_part[4][6];
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0)
        for (int d = 0; d < 3; ++d) { s_part[w][d] = mn[d]; s_part[w][3 + d] = mx[d]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        float r[6];
        for (int d = 0; d < 6; ++d) r[d] = s_part[0][d];
        for (int ww = 1; ww < 4; ++ww)
            for (int d = 0; d < 3; ++d) { r[d] = fmin_ref(r[d], s_part[ww][d]); r[3 + d] = fmax_ref(r[3 + d], s_part[ww][3 + d]); }
        for (int d = 0; d < 6; ++d) partials[blockIdx.x * 6 + d] = r[d];
    }
}

int launch_bbox(const float *x, const float *y, const float *z, int64_t n, float *partials, const FillSet &fills,
                hipStream_t s) {
    launch_more(fills, s);
    int64_t most = n;
    for (int f = 0; f < fills.k; ++f) most = fills.r[f].n > 4 * most ? fills.r[f].n / 4 : most;
    int64_t blocks = (most + 255) / 256;
    if (blocks > kBBoxBlocks) blocks = kBBoxBlocks;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_bbox, dim3((unsigned)blocks), dim3(256), 0, s, x, y, z, n, partials,
                       static_cast<const FillRanges &>(fills));
    return (int)blocks;
}

// ------------------------------------------------------------------ Morton
// toMortonCode / setMortonCodes (Solvers/MortonSort.h:46-73):
// (p - min) / maxSide, * 2^k, glm::clamp to [0, 2^k - 1], truncate,
// interleave as 4x + 2y + z.  NaN (zero-extent box) maps to 0.
__device__ __forceinline__ uint32_t quantize(float v, float mul, float hi) {
    float c = v * mul;
    float t = (c < 0.0f) ? 0.0f : c;      // glm::max(c, 0)
    t = (hi < t) ? hi : t;                // glm::min(t, hi)
    return (t != t) ? 0u : (uint32_t)t;
}

// Morton key of one point over the bounding cube of bb (min xyz, max xyz).
template <typename K>
__device__ __forceinline__ K morton_key(float px, float py, float pz, const float *bb) {
    const float mnx = bb[0], mny = bb[1], mnz = bb[2];
    const float dx = bb[3] - mnx, dy = bb[4] - mny, dz = bb[5] - mnz;
    const float m1 = (dx < dy) ? dy : dx;   // std::max(std::max(dx, dy), dz)
    const float scale = (m1 < dz) ? dz : m1;
    const float vx = ieee_div(px - mnx, scale);
    const float vy = ieee_div(py - mny, scale);
    const float vz = ieee_div(pz - mnz, scale);
    if constexpr (sizeof(K) == 4) {
        uint32_t qx = quantize(vx, 1024.0f, 1023.0f), qy = quantize(vy, 1024.0f, 1023.0f),
                 qz = quantize(vz, 1024.0f, 1023.0f);
        return expand_bits10(qx) * 4u + expand_bits10(qy) * 2u + expand_bits10(qz);
    } else {
        uint64_t qx = quantize(vx, 2097152.0f, 2097151.0f), qy = quantize(vy, 2097152.0f, 2097151.0f),
                 qz = quantize(vz, 2097152.0f, 2097151.0f);
        return expand_bits21(qx) * 4u + expand_bits21(qy) * 2u + expand_bits21(qz);
    }
}

// Keys, iota payload and the sort's digit histograms in one pass.  blocks >
// 0: the box is folded from k_bbox's partials and stored in bbox6;
// otherwise it is read from bbox6.
template <typename K>
__global__ __launch_bounds__(kKeyThreads) void k_morton(const float *__restrict__ x, const float *__restrict__ y,
                                                const float *__restrict__ z, int64_t n,
                                                const float *__restrict__ partials, int blocks, float *bbox6,
                                                K *__restrict__ keys, uint32_t *__restrict__ idx,
                                                uint32_t *__restrict__ ghist, int passes, int shift) {
    __shared__ uint32_t h[8 * kRadix];
    const DigitCount dc{h, passes, shift};
    dc.clear();
    float bb[6];
    if (blocks > 0) fold_bbox(partials, blocks, bb, bbox6);
    else
        for (int d = 0; d < 6; ++d) bb[d] = bbox6[d];
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const K k = morton_key<K>(x[i], y[i], z[i], bb);
        keys[i] = k;
        idx[i] = (uint32_t)i;
        dc.add(k);
    }
    __syncthreads();
    dc.store(ghist);
}

void launch_morton(const float *x, const float *y, const float *z, int64_t n, const float *partials, int blocks,
                   float *bbox6, int bits, const SortPlan &plan, void *keys, uint32_t *idx, void *keys_alt,
                   uint32_t *idx_alt, uint32_t *status, hipStream_t s) {
    if (n <= 0) return;
    const dim3 g(key_blocks(n)), t(key_threads(n));
    void *k = plan.from_alt ? keys_alt : keys;
    uint32_t *v = plan.from_alt ? idx_alt : idx;
    if (bits == 30)
        hipLaunchKernelGGL(k_morton<uint32_t>, g, t, 0, s, x, y, z, n, partials, blocks, bbox6,
                           (uint32_t *)k, v, status, plan.passes, plan.shift);
    else
        hipLaunchKernelGGL(k_morton<uint64_t>, g, t, 0, s, x, y, z, n, partials, blocks, bbox6,
                           (uint64_t *)k, v, status, plan.passes, plan.shift);
}

// ------------------------------------------------------------------ sort
// Stable LSD radix sort (8-bit digits), one "onesweep" kernel per pass:
// tiles take their index from an atomic counter, rank their keys in LDS with
// ballot-based digit matching (stable: wave-striped items in input order),
// publish per-digit tile counts, and resolve the global offset by decoupled
// look-back over earlier tiles.  Starting from an iota payload, the result
// is the order by (key, original index).
//
// Only the digits that a set of n keys needs to be told apart are sorted this
// way (sort_plan): spatial keys of n bodies differ in their top log2(n) + 10
// bits but for a few, and each pass is a launch that costs 7 us at least.  A
// last kernel moves every key to its place within the run of keys that share
// those bits, by its rank in the run (runs of one: a copy); runs of more than
// kRunMax keys (bodies much closer than the box suggests) are sorted by one
// workgroup each, up to run_one keys; past that all keys are sorted again by
// the whole grid.  Sort phase at 10,000 bodies 103 -> 30 us (63-bit keys),
// 170 -> 33 (octree paths, 102 bits), at 1,048,576 bodies 366 -> 122 (octree).
constexpr int64_t kRunMax = 256;
constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagPrefix = 2u << 30;
constexpr uint32_t kFlagMask = 3u << 30;
constexpr uint32_t kValueMask = (1u << 30) - 1;
constexpr uint32_t kSpinLimit = 1u << 22;

template <typename K>
__global__ __launch_bounds__(kSortBlock) void k_radix_hist(const K *__restrict__ keys, int64_t n, int passes, int shift,
                                                           uint32_t *__restrict__ ghist) {
    __shared__ uint32_t h[8 * kRadix];
    const DigitCount dc{h, passes, shift};
    dc.clear();
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dc.add(keys[i]);
    __syncthreads();
    dc.store(ghist);
}

// The LDS of a tile of NT threads with ITEMS keys each.
template <typename K, int NT, int ITEMS, bool SHARED>
struct TileLds {
    uint32_t wh[NT / kWave][kRadix];  // digit counts of the waves (cleared by the caller)
    uint32_t local_off[kRadix], gadj[kRadix], tmp[NT / kWave];
    K k[NT * ITEMS];
    uint32_t v[NT * ITEMS];
    uint8_t d[SHARED ? NT * ITEMS : 1];  // digits, where they come from the low words in memory
};

// Keys and payload that other workgroups write in the same kernel (SHARED) go
// past this XCD's caches.
template <bool SHARED, typename T>
__device__ __forceinline__ T sort_load(const T *p) {
    if constexpr (SHARED) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else return *p;
}
template <bool SHARED, typename T>
__device__ __forceinline__ void sort_store(T *p, T v) {
    if constexpr (SHARED) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}

// One tile of one pass: ghist holds the digits' counts over all keys, status
// the pass's look-back words.
template <typename K, int NT, int ITEMS, bool SHARED, typename Digit>
__device__ __forceinline__ void radix_tile(TileLds<K, NT, ITEMS, SHARED> &S, const K *kin, const uint32_t *vin, K *kout,
                                           uint32_t *vout, int64_t n, int64_t tile, const uint32_t *ghist,
                                           uint32_t *status, uint32_t *err, Digit &&digit) {
    constexpr int W = NT / kWave, TILE = NT * ITEMS;
    const int tid = threadIdx.x, lane = lane_id(), w = tid / kWave;
    const int64_t tile_base = tile * TILE;
    const int64_t wave_base = tile_base + (int64_t)w * (kWave * ITEMS);

    K key[ITEMS];
    uint32_t val[ITEMS], rnk[ITEMS], dig[SHARED ? ITEMS : 1];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int64_t i = wave_base + j * kWave + lane;
        if (i < n) { key[j] = sort_load<SHARED>(kin + i); val[j] = sort_load<SHARED>(vin + i); }
        else { key[j] = 0; val[j] = 0; }
    }
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const bool valid = (wave_base + j * kWave + lane) < n;
        const uint32_t d = digit(key[j], val[j]);
        if constexpr (SHARED) dig[j] = d;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            peers &= bit ? bb : ~bb;
        }
        uint32_t base = 0;
        if (valid) base = S.wh[w][d];
        const uint32_t below = __popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) S.wh[w][d] = base + __popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rnk[j] = base + below;
    }
    __syncthreads();

    // One thread per digit: exclusive prefix across waves, tile total.
    const uint32_t d = tid;
    const bool has = NT == kRadix || tid < kRadix;
    uint32_t tot = 0;
    if (has) {
#pragma unroll
        for (int ww = 0; ww < W; ++ww) {
            uint32_t c = S.wh[ww][d];
            S.wh[ww][d] = tot;
            tot += c;
        }
    }
    uint32_t *st = status + tile * kRadix;
    if (has) st_relaxed_agent(st + d, (tile == 0 ? kFlagPrefix : kFlagAgg) | tot);
    const uint32_t local_off = block_excl_scan<NT>(tot, S.tmp, nullptr);
    const uint32_t gbase = block_excl_scan<NT>(has ? sort_load<SHARED>(ghist + d) : 0u, S.tmp, nullptr);

    if (has) {
        uint32_t excl = 0;
        if (tile > 0) {
            int64_t p = tile - 1;
            uint32_t spins = 0;
            while (p >= 0) {
                const uint32_t sv = ld_acquire_agent(status + p * kRadix + d);
                const uint32_t f = sv & kFlagMask;
                if (f == 0) {
                    if (++spins > kSpinLimit) { atomicOr(err, 1u); break; }
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                excl += sv & kValueMask;
                if (f == kFlagPrefix) break;
                --p;
            }
            st_relaxed_agent(st + d, kFlagPrefix | (excl + tot));
        }
        S.local_off[d] = local_off;
        S.gadj[d] = gbase + excl - local_off;
    }
    __syncthreads();

#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const bool valid = (wave_base + j * kWave + lane) < n;
        if (valid) {
            uint32_t dj;
            if constexpr (SHARED) dj = dig[j];
            else dj = digit(key[j], val[j]);
            const uint32_t pos = S.local_off[dj] + S.wh[w][dj] + rnk[j];
            S.k[pos] = key[j];
            S.v[pos] = val[j];
            if constexpr (SHARED) S.d[pos] = (uint8_t)dj;
        }
    }
    __syncthreads();
    const int64_t rem = n - tile_base;
    const int ntile = rem < TILE ? (int)rem : TILE;
    for (int i = tid; i < ntile; i += NT) {
        const K k = S.k[i];
        const uint32_t v = S.v[i];
        uint32_t di;
        if constexpr (SHARED) di = S.d[i];
        else di = digit(k, v);
        const uint32_t g = S.gadj[di] + (uint32_t)i;
        if ((int64_t)g < n) {  // always true unless a look-back timed out
            sort_store<SHARED>(kout + g, k);
            sort_store<SHARED>(vout + g, v);
        } else {
            atomicOr(err, 1u);
        }
    }
}

template <typename K, int ITEMS>
__global__ __launch_bounds__(kSortBlock) void k_onesweep(const K *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                         K *__restrict__ kout, uint32_t *__restrict__ vout,
                                                         int64_t n, int shift, const uint32_t *__restrict__ ghist,
                                                         uint32_t *status, uint32_t *tile_counter, uint32_t *err) {
    __shared__ TileLds<K, kSortBlock, ITEMS, false> S;
    __shared__ uint32_t s_tile;
    if (threadIdx.x == 0) s_tile = atomicAdd(tile_counter, 1u);
    for (int i = threadIdx.x; i < kSortBlock / kWave * kRadix; i += kSortBlock) (&S.wh[0][0])[i] = 0;
    __syncthreads();
    radix_tile<K, kSortBlock, ITEMS, false>(S, kin, vin, kout, vout, n, s_tile, ghist, status, err,
                                            [&](K k, uint32_t) { return (uint32_t)(k >> shift) & 0xFFu; });
}

// The radix passes over bits shift .. shift + 8 passes - 1 (status cleared,
// histograms ready); the result is in the other buffer after an odd count.
template <typename K, int ITEMS>
static void radix_passes_i(K *ka, uint32_t *va, K *kb, uint32_t *vb, int64_t n, int passes, int shift,
                           uint32_t *status, uint32_t *err, hipStream_t s) {
    const int64_t tiles = (n + kSortBlock * ITEMS - 1) / (kSortBlock * ITEMS);
    uint32_t *ghist = status;                       // passes * 256
    uint32_t *counters = status + 8 * kRadix;       // passes; from + 32 on: long runs, the longest
    uint32_t *tstat = status + kSortHeadWords;      // passes * tiles * 256
    for (int p = 0; p < passes; ++p) {
        hipLaunchKernelGGL((k_onesweep<K, ITEMS>), dim3((unsigned)tiles), dim3(kSortBlock), 0, s, ka, va, kb, vb, n,
                           shift + 8 * p, ghist + p * kRadix, tstat + (int64_t)p * tiles * kRadix, counters + p, err);
        K *tk = ka; ka = kb; kb = tk;
        uint32_t *tv = va; va = vb; vb = tv;
    }
}

template <typename K>
static void radix_passes(K *ka, uint32_t *va, K *kb, uint32_t *vb, int64_t n, int passes, int shift, uint32_t *status,
                         uint32_t *err, hipStream_t s) {
    const int items = sort_items(n);
    if (items == 4) radix_passes_i<K, 4>(ka, va, kb, vb, n, passes, shift, status, err, s);
    else if (items == 8) radix_passes_i<K, 8>(ka, va, kb, vb, n, passes, shift, status, err, s);
    else radix_passes_i<K, 16>(ka, va, kb, vb, n, passes, shift, status, err, s);
}

// Low word of body v's key (an index out of range, which only a timed-out
// look-back leaves, and which k_sort_runs reports, has none).
__device__ __forceinline__ uint64_t low_word(const uint64_t *__restrict__ lo, uint32_t v, int64_t n) {
    return (int64_t)v < n ? lo[v] : 0ull;
}

// Whether key b at position j precedes key a at position i of a run sorted by
// prefix (both positions in the order of the original index).  lo: the low
// words of two-word keys, by original index.
template <typename K, bool LO>
__device__ __forceinline__ bool precedes(K b, uint32_t bi, int64_t j, K a, uint64_t alo, int64_t i,
                                         const uint64_t *__restrict__ lo, int64_t n) {
    if (b != a) return b < a;
    if (LO) {
        const uint64_t bl = low_word(lo, bi, n);
        if (bl != alo) return bl < alo;
    }
    return j < i;
}

// Moves the keys sorted by their bits from `shift` up (kin, vin) to their
// places by the whole key (kout, vout; lo_out: the low words in that order).
template <typename K, bool LO>
__global__ __launch_bounds__(256) void k_sort_runs(const K *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                   K *__restrict__ kout, uint32_t *__restrict__ vout, int64_t n,
                                                   int shift, const uint64_t *__restrict__ lo,
                                                   uint64_t *__restrict__ lo_out, uint32_t *nlong, uint32_t *longs,
                                                   uint32_t *err) {
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= n) return;
    const K a = kin[i], pre = a >> shift;
    const uint32_t v = vin[i];
    if ((int64_t)v >= n) { atomicOr(err, 1u); return; }  // only after a timed-out look-back
    uint64_t alo = 0;
    int64_t pos = i;
    const bool left = i > 0 && (kin[i - 1] >> shift) == pre, right = i + 1 < n && (kin[i + 1] >> shift) == pre;
    if (left || right) {
        // the run's ends, by galloping; of a long run, the end for its first key only
        int64_t b = i, e = i + 1;
        if (left) {
            int64_t out = -1;
            for (int64_t step = 1;; step *= 2) {
                const int64_t k = i - step;
                if (k < 0) break;
                if ((kin[k] >> shift) != pre) { out = k; break; }
                if (step >= kRunMax) return;  // long
                b = k;
            }
            while (b - out > 1) {
                const int64_t mid = out + (b - out) / 2;
                if ((kin[mid] >> shift) != pre) out = mid;
                else b = mid;
            }
        }
        if (right) {
            int64_t in = i, out = n;
            for (int64_t step = 1;; step *= 2) {
                const int64_t k = i + step;
                if (k >= n) break;
                if ((kin[k] >> shift) != pre) { out = k; break; }
                if (left && step >= kRunMax) return;
                in = k;
            }
            while (out - in > 1) {
                const int64_t mid = in + (out - in) / 2;
                if ((kin[mid] >> shift) != pre) out = mid;
                else in = mid;
            }
            e = out;
        }
        if (e - b > kRunMax) {
            if (i == b) {
                const uint32_t slot = atomicAdd(nlong, 1u);
                atomicMax(nlong + 1, (uint32_t)(e - b));
                if (slot < kSortLongRuns) {
                    longs[2 * slot] = (uint32_t)b;
                    longs[2 * slot + 1] = (uint32_t)(e - b);
                }
            }
            return;
        }
        pos = b;
        if (LO) alo = lo[v];
        for (int64_t j = b; j < e; ++j) pos += precedes<K, LO>(kin[j], vin[j], j, a, alo, i, lo, n) ? 1 : 0;
    }
    kout[pos] = a;
    vout[pos] = v;
    if (LO) lo_out[pos] = left || right ? alo : lo[v];
}

// Every key again, by the whole key, in one kernel: where a run is long, most
// keys share the bits that the passes sorted by, and one workgroup's time with
// it would grow with the run.  Sort phase, ms, of 1,000,000 bodies of which two
// are 1,000 / 10,000 radii out, a workgroup a run and so: linear BVH 0.90 /
// 2.80 -> 0.50 / 0.47, octree 2.65 / 4.06 -> 0.78 / 0.73.  The digit counts,
// the radix passes (but for digits that all keys share) and the copy to the
// output are stages of `tiles` tasks each, handed out by one counter in that
// order; a stage takes some 40 us at that size, of which the look-back and
// the fences are most.  A task waits for the stage before it, whose tasks
// were all handed out earlier, to workgroups that run: no workgroup waits for
// one that has not started, however few are on the GPU at a time.
constexpr int kAllItems = 4, kAllTile = 1024 * kAllItems;
template <typename K>
using AllLds = TileLds<K, 1024, kAllItems, true>;

template <typename K, bool LO>
__device__ void sort_all(AllLds<K> &S, K *ka, uint32_t *va, K *kb, uint32_t *vb, int64_t n,
                         const uint64_t *__restrict__ lo, uint64_t *__restrict__ lo_out, uint32_t *words,
                         uint32_t *tstat, uint32_t *err) {
    __shared__ uint32_t s_task, s_late, s_equal;  // s_equal: passes whose digit all keys share
    constexpr int kLowPasses = LO ? 5 : 0, kPasses = kLowPasses + (int)sizeof(K);
    static_assert(kPasses <= kSortAllPasses, "words for the counts");
    uint32_t *ghist = words, *next = words + kSortAllPasses * kRadix, *done = next + 1;
    const int tid = threadIdx.x;
    const uint32_t tiles = (uint32_t)((n + kAllTile - 1) / kAllTile);
    // the look-back words of three passes in turn: the next pass's are cleared
    // while those of the pass before are no longer read
    auto status_of = [&](int pass) { return tstat + (int64_t)(pass % 3) * tiles * kRadix; };
    if (tid == 0) s_equal = 0;
    bool counted = false;
    int passes = kPasses;
    for (;;) {
        __syncthreads();
        if (tid == 0) s_task = atomicAdd(next, 1u);
        __syncthreads();
        const uint32_t stage = s_task / tiles, tile = s_task % tiles;
        if (stage > (uint32_t)passes + 1) return;
        auto wait_for = [&](uint32_t before) {  // false: given up
            if (tid == 0) {
                uint32_t spins = 0;
                s_late = 0;
                while (ld_acquire_agent(done + before) < tiles) {
                    if (++spins > kSpinLimit) { atomicOr(err, 1u); s_late = 1; break; }
                    __builtin_amdgcn_s_sleep(8);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // for the workgroup, with the barriers around it
            }
            __syncthreads();
            return s_late == 0;
        };
        if (stage > 0 && !counted) {
            if (!wait_for(0)) return;
            for (int i = tid; i < kPasses * kRadix; i += 1024)
                if (sort_load<true>(ghist + i) == (uint32_t)n) atomicOr(&s_equal, 1u << (i / kRadix));
            __syncthreads();
            counted = true;
            passes = kPasses - __popc(s_equal);
            if (stage > (uint32_t)passes + 1) return;
        }
        if (stage > 1 && !wait_for(stage - 1)) return;
        const int64_t base = (int64_t)tile * kAllTile, end = base + kAllTile < n ? base + kAllTile : n;
        auto digit = [&](int pass, K k, uint32_t v) {
            return pass < kLowPasses ? (uint32_t)(low_word(lo, v, n) >> (8 * pass)) & 0xFFu
                                     : (uint32_t)(k >> (8 * (pass - kLowPasses))) & 0xFFu;
        };
        if (stage <= (uint32_t)passes && tid < kRadix) st_relaxed_agent(status_of(stage) + tile * kRadix + tid, 0u);
        if (stage == 0) {
            uint32_t *h = reinterpret_cast<uint32_t *>(S.k);
            static_assert(sizeof S.k >= kPasses * kRadix * 4, "the counts' place");
            for (int i = tid; i < kPasses * kRadix; i += 1024) h[i] = 0;
            __syncthreads();
            for (int64_t i0 = base; i0 < end; i0 += 1024) {
                const int64_t i = i0 + tid;
                const bool ok = i < end;
                const K k = ok ? ka[i] : K(0);
                const uint32_t v = ok ? va[i] : 0u;
                const uint64_t low = LO && ok ? low_word(lo, v, n) : 0ull;
                const uint64_t in = __ballot(ok);
                for (int p = 0; p < kPasses; ++p) {
                    const uint32_t d = p < kLowPasses ? (uint32_t)(low >> (8 * p)) & 0xFFu
                                                      : (uint32_t)(k >> (8 * (p - kLowPasses))) & 0xFFu;
                    // most waves' keys share most digits: one addition for them all
                    const uint32_t first = (uint32_t)uniform_i32((int)d);
                    const bool same = __ballot(ok && d == first) == in;
                    if (same ? lane_id() == 0 && in : ok) atomicAdd(&h[p * kRadix + d], same ? (uint32_t)__popcll(in) : 1u);
                }
            }
            __syncthreads();
            for (int i = tid; i < kPasses * kRadix; i += 1024)
                if (h[i]) atomicAdd(&ghist[i], h[i]);
        } else if (stage <= (uint32_t)passes) {
            const int step = (int)stage - 1;
            uint32_t todo = ((1u << kPasses) - 1u) & ~s_equal;
            for (int k = 0; k < step; ++k) todo &= todo - 1;
            const int p = __builtin_ctz(todo);
            for (int i = tid; i < 1024 / kWave * kRadix; i += 1024) (&S.wh[0][0])[i] = 0;
            __syncthreads();
            const bool back = step & 1;
            radix_tile<K, 1024, kAllItems, true>(S, back ? kb : ka, back ? vb : va, back ? ka : kb, back ? va : vb, n,
                                                 tile, ghist + p * kRadix, status_of(step), err,
                                                 [&](K k, uint32_t v) { return digit(p, k, v); });
        } else {
            for (int64_t i = base + tid; i < end; i += 1024) {
                const uint32_t v = sort_load<true>((passes & 1 ? vb : va) + i);
                if (!(passes & 1)) {
                    kb[i] = sort_load<true>(ka + i);
                    vb[i] = v;
                }
                if (LO) lo_out[i] = low_word(lo, v, n);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's stores have arrived
        __syncthreads();
        if (tid == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            atomicAdd(done + stage, 1u);
        }
    }
}

// The runs that k_sort_runs left: one workgroup sorts one run at a time by its
// low digits (LSD, stable), the run's two buffers in turn.  More long runs
// than the list holds: every workgroup looks for the runs' heads itself.  A
// run of more than run_one keys: all keys are sorted again (sort_all, 100 to
// 300 us below 100,000 keys; one workgroup takes 10 us for each 1,024 keys of
// the longest run, 25 with low words).
constexpr uint32_t run_one(bool lo) { return lo ? 4096 : 16384; }
template <typename K, bool LO>
__global__ __launch_bounds__(1024) void k_sort_long(K *__restrict__ kin, uint32_t *__restrict__ vin,
                                                    K *__restrict__ kout, uint32_t *__restrict__ vout, int64_t n,
                                                    int shift, const uint64_t *__restrict__ lo,
                                                    uint64_t *__restrict__ lo_out, const uint32_t *nlong,
                                                    const uint32_t *longs, uint32_t *words, uint32_t *tstat,
                                                    uint32_t *err) {
    constexpr int W = 1024 / kWave;
    __shared__ uint32_t cnt[kRadix], wh[W][kRadix], tmp[W];
    __shared__ int unsorted;
    const uint32_t runs = nlong[0];
    if (runs == 0) return;
    if (nlong[1] > run_one(LO)) {
        __shared__ AllLds<K> S;
        sort_all<K, LO>(S, kin, vin, kout, vout, n, lo, lo_out, words, tstat, err);
        return;
    }
    const int tid = threadIdx.x, lane = lane_id(), w = tid / kWave;
    auto sort_run = [&](int64_t b, int64_t m) {
        // already in order (coincident bodies): a copy
        if (tid == 0) unsorted = 0;
        __syncthreads();
        bool bad = false;
        for (int64_t i = tid; i + 1 < m; i += 1024) {
            const K k0 = kin[b + i], k1 = kin[b + i + 1];
            if (k0 > k1 || (LO && k0 == k1 && low_word(lo, vin[b + i], n) > low_word(lo, vin[b + i + 1], n))) bad = true;
        }
        if (bad) unsorted = 1;
        __syncthreads();
        K *ka = kin + b, *kb = kout + b;
        uint32_t *va = vin + b, *vb = vout + b;
        const int plo = LO ? 5 : 0, passes = unsorted ? plo + (shift + 7) / 8 : 0;
        for (int p = 0; p < passes; ++p) {
            auto digit = [&](K k, uint32_t v) {
                return p < plo ? (uint32_t)(low_word(lo, v, n) >> (8 * p)) & 0xFFu : (uint32_t)(k >> (8 * (p - plo))) & 0xFFu;
            };
            if (tid < kRadix) cnt[tid] = 0;
            __syncthreads();
            for (int64_t i = tid; i < m; i += 1024) atomicAdd(&cnt[digit(ka[i], va[i])], 1u);
            __syncthreads();
            const uint32_t c = tid < kRadix ? cnt[tid] : 0u;
            const uint32_t ex = block_excl_scan<1024>(c, tmp, nullptr);
            if (tid < kRadix) cnt[tid] = ex;
            for (int64_t t0 = 0; t0 < m; t0 += 1024) {
                for (int i = tid; i < W * kRadix; i += 1024) (&wh[0][0])[i] = 0;
                __syncthreads();
                const bool ok = t0 + tid < m;
                K k = 0;
                uint32_t v = 0, d = 0;
                if (ok) { k = ka[t0 + tid]; v = va[t0 + tid]; d = digit(k, v); }
                uint64_t peers = __ballot(ok);
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const uint64_t bb = __ballot((d >> q) & 1u);
                    peers &= ((d >> q) & 1u) ? bb : ~bb;
                }
                const uint32_t below = __popcll(peers & lanemask_lt());
                if (ok && below == 0) wh[w][d] = (uint32_t)__popcll(peers);
                __syncthreads();
                if (tid < kRadix) {
                    uint32_t run = cnt[tid];
                    for (int q = 0; q < W; ++q) {
                        const uint32_t x = wh[q][tid];
                        wh[q][tid] = run;
                        run += x;
                    }
                    cnt[tid] = run;
                }
                __syncthreads();
                if (ok) {
                    const uint32_t o = wh[w][d] + below;
                    kb[o] = k;
                    vb[o] = v;
                }
                __syncthreads();
            }
            K *tk = ka; ka = kb; kb = tk;
            uint32_t *tv = va; va = vb; vb = tv;
            __threadfence_block();
            __syncthreads();
        }
        if (ka != kout + b)
            for (int64_t i = tid; i < m; i += 1024) { kout[b + i] = ka[i]; vout[b + i] = va[i]; }
        __syncthreads();
        if (LO)
            for (int64_t i = tid; i < m; i += 1024) lo_out[b + i] = low_word(lo, vout[b + i], n);
        __syncthreads();
        (void)lane;
    };
    if (runs <= (uint32_t)kSortLongRuns) {
        for (uint32_t r = blockIdx.x; r < runs; r += gridDim.x) {
            const int64_t b = longs[2 * r], m = longs[2 * r + 1];
            if (b + m <= n) sort_run(b, m);
        }
        return;
    }
    // the list overflowed: heads by position, kRunMax apart at least
    __shared__ int64_t head, len;
    for (int64_t c = blockIdx.x; c * kRunMax < n; c += gridDim.x) {
        // a long run's head in [c kRunMax, (c + 1) kRunMax): at most one
        __syncthreads();
        if (tid == 0) head = -1;
        __syncthreads();
        const int64_t i = c * kRunMax + tid;
        if (tid < kRunMax && i + kRunMax < n) {
            const K pre = kin[i] >> shift;
            if ((i == 0 || (kin[i - 1] >> shift) != pre) && (kin[i + kRunMax] >> shift) == pre) {
                int64_t in = i + kRunMax, out = n;
                while (out - in > 1) {
                    const int64_t mid = in + (out - in) / 2;
                    if ((kin[mid] >> shift) != pre) out = mid;
                    else in = mid;
                }
                head = i;
                len = out - i;
            }
        }
        __syncthreads();
        const int64_t hb = head, hl = len;
        if (hb >= 0) sort_run(hb, hl);
    }
}

template <typename K>
static void sort_planned(K *keys, uint32_t *idx, K *keys_alt, uint32_t *idx_alt, int64_t n, const SortPlan &plan,
                         const uint64_t *lo, uint64_t *lo_sorted, uint32_t *status, uint32_t *err, hipStream_t s) {
    K *ka = plan.from_alt ? keys_alt : keys, *kb = plan.from_alt ? keys : keys_alt;
    uint32_t *va = plan.from_alt ? idx_alt : idx, *vb = plan.from_alt ? idx : idx_alt;
    radix_passes(ka, va, kb, vb, n, plan.passes, plan.shift, status, err, s);
    if (!plan.runs) return;
    uint32_t *nlong = status + 8 * kRadix + 32, *longs = status + 8 * kRadix + 64, *words = longs + 2 * kSortLongRuns;
    const dim3 g((unsigned)((n + 255) / 256));
    const unsigned gl = n <= kRunMax ? 0u : (unsigned)(n / kRunMax < 256 ? n / kRunMax : 256);
    if (lo) {
        hipLaunchKernelGGL((k_sort_runs<K, true>), g, dim3(256), 0, s, keys_alt, idx_alt, keys, idx, n, plan.shift, lo,
                           lo_sorted, nlong, longs, err);
        if (gl)
            hipLaunchKernelGGL((k_sort_long<K, true>), dim3(gl), dim3(1024), 0, s, keys_alt, idx_alt, keys, idx, n,
                               plan.shift, lo, lo_sorted, nlong, longs, words, status + kSortHeadWords, err);
    } else {
        hipLaunchKernelGGL((k_sort_runs<K, false>), g, dim3(256), 0, s, keys_alt, idx_alt, keys, idx, n, plan.shift, lo,
                           lo_sorted, nlong, longs, err);
        if (gl)
            hipLaunchKernelGGL((k_sort_long<K, false>), dim3(gl), dim3(1024), 0, s, keys_alt, idx_alt, keys, idx, n,
                               plan.shift, lo, lo_sorted, nlong, longs, words, status + kSortHeadWords, err);
    }
}

void launch_sort(void *keys, uint32_t *idx, void *keys_alt, uint32_t *idx_alt, int64_t n, int bits,
                 const SortPlan &plan, uint32_t *status, uint32_t *err, hipStream_t s, const uint64_t *lo,
                 uint64_t *lo_sorted) {
    if (n <= 0) return;
    if (bits == 30)
        sort_planned<uint32_t>((uint32_t *)keys, idx, (uint32_t *)keys_alt, idx_alt, n, plan, nullptr, nullptr, status,
                               err, s);
    else
        sort_planned<uint64_t>((uint64_t *)keys, idx, (uint64_t *)keys_alt, idx_alt, n, plan, lo, lo_sorted, status,
                               err, s);
}

bool launch_radix_sort_u64(uint64_t *keys, uint32_t *idx, uint64_t *keys_alt, uint32_t *idx_alt, int64_t n,
                           int passes, uint32_t *status, uint32_t *err, hipStream_t s) {
    if (n <= 1 || passes <= 0) return false;
    launch_fill_u32(status, 0u, kSortHeadWords + passes * sort_tiles(n) * kRadix, s);
    int64_t hb = (n + 4095) / 4096;
    if (hb > 2048) hb = 2048;
    hipLaunchKernelGGL(k_radix_hist<uint64_t>, dim3((unsigned)hb), dim3(kSortBlock), 0, s, keys, n, passes, 0, status);
    radix_passes(keys, idx, keys_alt, idx_alt, n, passes, 0, status, err, s);
    return (passes & 1) != 0;
}

// ------------------------------------------------------------------ gather
__global__ __launch_bounds__(256) void k_gather(const float *__restrict__ x, const float *__restrict__ y,
                                                const float *__restrict__ z, const float *__restrict__ m,
                                                const uint32_t *__restrict__ perm, int64_t n,
                                                float4 *__restrict__ bodies) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t j = perm[i];
        bodies[i] = (int64_t)j < n ? make_float4(x[j], y[j], z[j], m[j]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

void launch_gather(const float *x, const float *y, const float *z, const float *m, const uint32_t *perm,
                   int64_t n, float4 *bodies, hipStream_t s) {
    if (n <= 0) return;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_gather, dim3((unsigned)blocks), dim3(256), 0, s, x, y, z, m, perm, n, bodies);
}

// ------------------------------------------------------------------ LBVH topology
// Karras (2012) radix tree over the sorted keys with index-augmented key
// comparison.  For a range whose end keys differ, the Karras split is the
// first index whose key has the highest differing bit set, i.e. exactly
// LinearBVHNode::split (Trees/LinearBVH.h:47-76).  The reference stops
// splitting at size <= leaf or all-equal keys (LinearBVH.h:114-119); since a
// splittable node's ancestors are splittable too, the reference tree is the
// root plus the children of the splittable Karras nodes.
template <typename K>
__device__ __forceinline__ int kdelta(const K *__restrict__ keys, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const K a = keys[i], b = keys[j];
    if (a == b) return (int)(8 * sizeof(K)) + __clz((uint32_t)(i ^ j));
    if constexpr (sizeof(K) == 8) return __clzll((unsigned long long)(a ^ b));
    else return __clz((uint32_t)(a ^ b));
}

// Forest (sys_shift > 0): keys carry the system index above bit sys_shift; a
// node whose range spans systems always splits, and a node inside system s
// uses that system's leaf size leaf_tab[s].
template <typename K>
__global__ __launch_bounds__(256) void k_karras(const K *__restrict__ keys, int n, int leaf, int32_t *kfirst,
                                                int32_t *klast, int32_t *kgamma, uint32_t *ksplit,
                                                int32_t *kparent, uint32_t *sums, int sys_shift,
                                                const int32_t *__restrict__ leaf_tab) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (kdelta(keys, n, i, i + 1) - kdelta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = kdelta(keys, n, i, i - d);
    int lmax = 2;
    while (kdelta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (kdelta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = kdelta(keys, n, i, j);
    int sp = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (kdelta(keys, n, i, i + (sp + t) * d) > dnode) sp += t;
    } while (t > 1);
    const int gamma = i + sp * d + (d < 0 ? -1 : 0);
    const int first = d > 0 ? i : j, last = d > 0 ? j : i;
    kfirst[i] = first;
    klast[i] = last;
    kgamma[i] = gamma;
    int L = leaf;
    bool span = false;
    if (sys_shift > 0) {
        const uint64_t s0 = (uint64_t)keys[first] >> sys_shift, s1 = (uint64_t)keys[last] >> sys_shift;
        span = s0 != s1;
        L = leaf_tab[s0];
    }
    const uint32_t split = ((span || last - first + 1 > L) && keys[first] != keys[last]) ? 1u : 0u;
    ksplit[i] = split;
    scan_sum(split, i, sums);
    if (gamma != first) kparent[gamma] = 2 * i;
    if (gamma + 1 != last) kparent[gamma + 1] = 2 * i + 1;
}

// Exclusive scan of u32 flags: each tile's sum (added up by the kernel that
// computes the flags, scan_sum, or by one of its own), then the tiles.
__global__ __launch_bounds__(kScanBlock) void k_scan_top(uint32_t *sums, int64_t nt, uint32_t *total) {
    __shared__ uint32_t s_tmp[kScanBlock / kWave];
    uint32_t carry = 0;
    for (int64_t b = 0; b < nt; b += kScanBlock) {
        int64_t i = b + threadIdx.x;
        uint32_t v = i < nt ? sums[i] : 0u;
        uint32_t tot;
        uint32_t e = block_excl_scan<kScanBlock>(v, s_tmp, &tot);
        if (i < nt) sums[i] = carry + e;
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

// in may equal out: every thread reads its items before it writes them.
// FOLD: sums still holds the tiles' own sums, and every workgroup adds up
// those before it (at most kScanFold tiles: one launch less than a scan of
// the sums, 4 us of a small build); the last tile stores the total.
// nlim (or null): a device count of items; those from *nlim on are zero.
template <bool FOLD>
__global__ __launch_bounds__(kScanBlock) void k_scan_tiles(const uint32_t *in, int64_t n, const uint32_t *nlim,
                                                           const uint32_t *__restrict__ sums, uint32_t *out,
                                                           uint32_t *total) {
    __shared__ uint32_t s_tmp[kScanBlock / kWave];
    const int64_t base = blockIdx.x * (int64_t)kScanTile;
    uint32_t before = 0;
    if (FOLD) {
        uint32_t acc = 0;
        for (unsigned t = threadIdx.x; t < blockIdx.x; t += kScanBlock) acc += sums[t];
        block_excl_scan<kScanBlock>(acc, s_tmp, &before);
        if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = before + sums[blockIdx.x];
    } else {
        before = sums[blockIdx.x];
    }
    const int64_t lim = nlim && (int64_t)*nlim < n ? (int64_t)*nlim : n;
    if (base >= lim) return;  // nothing reads past the items
    // Blocked arrangement: thread t owns items [t*I, t*I + I).
    uint32_t v[kScanItems], acc = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        int64_t i = base + (int64_t)threadIdx.x * kScanItems + j;
        v[j] = i < lim ? in[i] : 0u;
        acc += v[j];
    }
    uint32_t run = before + block_excl_scan<kScanBlock>(acc, s_tmp, nullptr);
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        int64_t i = base + (int64_t)threadIdx.x * kScanItems + j;
        if (i < lim) out[i] = run;
        run += v[j];
    }
}

__global__ __launch_bounds__(kScanBlock) void k_scan_sums(const uint32_t *__restrict__ in, int64_t n,
                                                          const uint32_t *nlim, uint32_t *__restrict__ sums) {
    __shared__ uint32_t s_tmp[kScanBlock / kWave];
    const int64_t base = blockIdx.x * (int64_t)kScanTile;
    const int64_t lim = nlim && (int64_t)*nlim < n ? (int64_t)*nlim : n;
    uint32_t acc = 0;
    for (int j = 0; j < kScanItems; ++j) {
        const int64_t i = base + (int64_t)j * kScanBlock + threadIdx.x;
        if (i < lim) acc += in[i];
    }
    uint32_t tot;
    block_excl_scan<kScanBlock>(acc, s_tmp, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

void launch_scan_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *sums, uint32_t *total, hipStream_t s,
                     const uint32_t *nlim) {
    const int64_t nt = (n + kScanTile - 1) / kScanTile;
    const dim3 g((unsigned)nt), t(kScanBlock);
    if (!scan_fused(n)) hipLaunchKernelGGL(k_scan_sums, g, t, 0, s, in, n, nlim, sums);
    if (nt <= kScanFold) {
        hipLaunchKernelGGL(k_scan_tiles<true>, g, t, 0, s, in, n, nlim, sums, out, total);
        return;
    }
    hipLaunchKernelGGL(k_scan_top, dim3(1), t, 0, s, sums, nt, total);
    hipLaunchKernelGGL(k_scan_tiles<false>, g, t, 0, s, in, n, nlim, sums, out, total);
}

// The compact nodes, the node count, and the bodies in key order.
__global__ __launch_bounds__(256) void k_emit(int n, const int32_t *__restrict__ kfirst,
                                              const int32_t *__restrict__ klast, const int32_t *__restrict__ kgamma,
                                              const uint32_t *__restrict__ ksplit, const uint32_t *__restrict__ krank,
                                              const int32_t *__restrict__ kparent,
                                              const uint32_t *__restrict__ total, NodeRec *__restrict__ nodes,
                                              int32_t *__restrict__ leaf_start, uint32_t *__restrict__ node_count,
                                              const float *__restrict__ x, const float *__restrict__ y,
                                              const float *__restrict__ z, const float *__restrict__ m,
                                              const uint32_t *__restrict__ perm, float4 *__restrict__ bodies) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = perm[i];
    bodies[i] = j < (uint32_t)n ? make_float4(x[j], y[j], z[j], m[j]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (i == 0) {
        const bool inner = n > 1 && ksplit[0];
        if (!inner) {
            nodes[0].topo = make_int4(0, n, -1, -1);
            leaf_start[0] = 0;
        }
        *node_count = inner ? 1u + 2u * *total : 1u;
    }
    if (i >= n - 1 || !ksplit[i]) return;
    const int r = (int)krank[i];
    const int first = kfirst[i], last = klast[i], gamma = kgamma[i];
    int my_slot = 0;
    if (i != 0) {
        const int pk = kparent[i];
        my_slot = 1 + 2 * (int)krank[pk >> 1] + (pk & 1);
    } else {
        nodes[0].topo = make_int4(first, last - first + 1, 1 + 2 * r, -1);
    }
    const int kl = gamma, kr = gamma + 1;
    const bool l_int = (gamma != first), r_int = (gamma + 1 != last);
    const int lptr = (l_int && ksplit[kl]) ? 1 + 2 * (int)krank[kl] : -1;
    const int rptr = (r_int && ksplit[kr]) ? 1 + 2 * (int)krank[kr] : -1;
    nodes[1 + 2 * r].topo = make_int4(first, gamma - first + 1, lptr, my_slot);
    nodes[2 + 2 * r].topo = make_int4(gamma + 1, last - gamma, rptr, my_slot);
    if (lptr < 0) leaf_start[first] = 1 + 2 * r;
    if (rptr < 0) leaf_start[gamma + 1] = 2 + 2 * r;
}

void launch_lbvh_topology(const void *keys, int bits, int64_t n64, int leaf_size, int32_t *kfirst, int32_t *klast,
                          int32_t *kgamma, uint32_t *ksplit, uint32_t *krank, int32_t *kparent, uint32_t *scan_ws,
                          NodeRec *nodes, int32_t *leaf_start, uint32_t *node_count, const float *x, const float *y,
                          const float *z, const float *m, const uint32_t *perm, float4 *bodies, hipStream_t s,
                          int sys_shift, const int32_t *leaf_tab) {
    if (n64 <= 0) {
        launch_fill_u32(node_count, 0u, 1, s);
        return;
    }
    const int n = (int)n64;
    uint32_t *total = scan_ws, *sums = scan_ws + 64;
    const dim3 g((unsigned)((n + 255) / 256)), t(256);
    if (n >= 2) {
        const int k = n - 1;
        const dim3 gk((unsigned)((k + 255) / 256));
        uint32_t *fused = scan_fused(k) ? sums : nullptr;
        if (bits == 30)
            hipLaunchKernelGGL(k_karras<uint32_t>, gk, t, 0, s, (const uint32_t *)keys, n, leaf_size, kfirst, klast,
                               kgamma, ksplit, kparent, fused, 0, (const int32_t *)nullptr);
        else
            hipLaunchKernelGGL(k_karras<uint64_t>, gk, t, 0, s, (const uint64_t *)keys, n, leaf_size, kfirst, klast,
                               kgamma, ksplit, kparent, fused, sys_shift, leaf_tab);
        launch_scan_u32(ksplit, krank, k, sums, total, s);
    }
    hipLaunchKernelGGL(k_emit, g, t, 0, s, n, kfirst, klast, kgamma, ksplit, krank, kparent, total, nodes, leaf_start,
                       node_count, x, y, z, m, perm, bodies);
}

// ------------------------------------------------------------------ summaries
// NodeBase::summarize (Trees/NodeBase.h:43-55) bottom-up.  A leaf takes
// CenterOfMassSummary's sequential sums over its bodies in sort order
// (Summaries/CenterOfMassSummary.h:30-42) and its bounding box
// (Summaries/BoundingBoxSummary.h:30-57); an internal node combines its two
// children (CenterOfMassSummary.h:44-55, BoundingBoxSummary.h:59-68).  The
// combine reads only finished children, so the result does not depend on
// which child finishes first.  The MAC record is (bbox centre (max+min)/2,
// |max-min|^2) (Physics/BoundingBox.h:47,55).
//
// Scheduling: a chain of dependent steps from the deepest leaf to the root,
// so what counts is the time of one step.  Each workgroup owns a range of
// consecutive bodies.  Its threads summarise the leaves that start in it and
// climb: the two children of a node meet in LDS (the place of the meeting is
// the split position between them), the first to arrive leaves its summary
// and stops, the second takes both on to the parent.  A node whose parent
// leaves the range is queued, and the next launch climbs on from the queue
// with ranges 32 times as long, the last one without ranges.  Meeting in LDS
// instead of through arrival counters and records in memory: 10,000 bodies
// (63-bit keys) 148 -> 53 us, 500,000 bodies 210 -> 130, 1,048,576 bodies
// (30-bit keys) 188 -> 159.  Bound by the chain: about 1 us a level.
// The MAC record: bbox centre and the squared-distance threshold above which
// a target accepts the node (mac_lbvh_threshold of the squared diagonal).
// Per-node choice of the MAC parameters: one set, or per system of a forest
// (the system index is the key prefix of the node's first body).
struct MacSel {
    MacParam one;
    const MacParam *tab;
    const uint64_t *keys;
    int shift;
    __device__ __forceinline__ MacParam at(int first) const { return tab ? tab[keys[first] >> shift] : one; }
    // Forest: a node whose range spans systems needs no summary (every walk
    // starts at a system's root), so climbs stop below it.
    __device__ __forceinline__ bool spans(int4 t) const {
        return tab && (keys[t.x] >> shift) != (keys[t.x + t.y - 1] >> shift);
    }
};

__device__ __forceinline__ float4 mac_record(float4 mn, float4 mx, MacParam mp) {
    const float cx = (mx.x + mn.x) / 2.0f, cy = (mx.y + mn.y) / 2.0f, cz = (mx.z + mn.z) / 2.0f;
    const float dx = mx.x - mn.x, dy = mx.y - mn.y, dz = mx.z - mn.z;
    const float diag2 = dx * dx + dy * dy + dz * dz;
    return make_float4(cx, cy, cz, mac_lbvh_threshold(diag2, mp.mid, mp.tie != 0));
}

// A node's summary while a thread climbs: its parent's is made from it and
// the sibling's, which alone is then read from memory.
struct LbvhSum {
    float4 com, mn, mx;
};

__device__ __forceinline__ LbvhSum summarize_leaf(int4 t, const float4 *__restrict__ bodies) {
    float M = 0.0f, cx = 0.0f, cy = 0.0f, cz = 0.0f;
    float nx = FLT_MAX, ny = FLT_MAX, nz = FLT_MAX, xx = -FLT_MAX, xy = -FLT_MAX, xz = -FLT_MAX;
    auto add = [&](float4 b) {
        M += b.w;
        cx = cx + b.x * b.w;
        cy = cy + b.y * b.w;
        cz = cz + b.z * b.w;
        nx = fmin_ref(b.x, nx); ny = fmin_ref(b.y, ny); nz = fmin_ref(b.z, nz);
        xx = fmax_ref(b.x, xx); xy = fmax_ref(b.y, xy); xz = fmax_ref(b.z, xz);
    };
    // four loads in flight; the sums stay sequential
    int i = t.x;
    for (; i + 4 <= t.x + t.y; i += 4) {
        const float4 b0 = bodies[i], b1 = bodies[i + 1], b2 = bodies[i + 2], b3 = bodies[i + 3];
        add(b0); add(b1); add(b2); add(b3);
    }
    for (; i < t.x + t.y; ++i) add(bodies[i]);
    LbvhSum r;
    r.com = make_float4(ieee_div(cx, M), ieee_div(cy, M), ieee_div(cz, M), M);
    r.mn = make_float4(nx, ny, nz, 0.0f);
    r.mx = make_float4(xx, xy, xz, 0.0f);
    return r;
}

__device__ __forceinline__ LbvhSum summarize_pair(const LbvhSum &a, const LbvhSum &b) {
    LbvhSum r;
    float Mp = 0.0f;
    Mp += a.com.w;
    float px = 0.0f + a.com.x * a.com.w, py = 0.0f + a.com.y * a.com.w, pz = 0.0f + a.com.z * a.com.w;
    Mp += b.com.w;
    px = px + b.com.x * b.com.w;
    py = py + b.com.y * b.com.w;
    pz = pz + b.com.z * b.com.w;
    r.com = make_float4(ieee_div(px, Mp), ieee_div(py, Mp), ieee_div(pz, Mp), Mp);
    const float4 n0 = make_float4(fmin_ref(a.mn.x, FLT_MAX), fmin_ref(a.mn.y, FLT_MAX), fmin_ref(a.mn.z, FLT_MAX), 0.0f);
    const float4 x0 =
        make_float4(fmax_ref(a.mx.x, -FLT_MAX), fmax_ref(a.mx.y, -FLT_MAX), fmax_ref(a.mx.z, -FLT_MAX), 0.0f);
    r.mn = make_float4(fmin_ref(b.mn.x, n0.x), fmin_ref(b.mn.y, n0.y), fmin_ref(b.mn.z, n0.z), 0.0f);
    r.mx = make_float4(fmax_ref(b.mx.x, x0.x), fmax_ref(b.mx.y, x0.y), fmax_ref(b.mx.z, x0.z), 0.0f);
    return r;
}

__device__ __forceinline__ void store_sum(int s, const LbvhSum &v, NodeRec *nodes, float4 *bmin, float4 *bmax) {
    nodes[s].com = v.com;
    bmin[s] = v.mn;
    bmax[s] = v.mx;
}

// MultipoleMassSummary::summarize(childNodes) (MultipoleMassSummary.h:54-65)
// for two children: (0 + t0) + t1 with t = outer(c_child - c, c_child) m_child
// + Q_child.
__device__ __forceinline__ void quad_pair(float4 c, float4 a, const float qa[6], float4 b, const float qb[6], float Q[6]) {
    float t[6], u[6];
    quad_term(a.x - c.x, a.y - c.y, a.z - c.z, a.w, t);
    quad_term(b.x - c.x, b.y - c.y, b.z - c.z, b.w, u);
#pragma unroll
    for (int e = 0; e < 6; ++e) Q[e] = (0.0f + (t[e] + qa[e])) + (u[e] + qb[e]);
}

// What a pass of the climb works on.
struct SummPass {
    NodeRec *nodes;
    float4 *bmin, *bmax, *quad;
    int64_t n, max_nodes;
    uint32_t *flags;    // arrival counters by node, for passes whose meetings outgrow LDS
    // queue of the nodes whose parent leaves the range (null: no ranges): each
    // workgroup's from its first body's position on, and their number
    uint32_t *qout, *qout_n;
    MacSel ms;
    uint32_t *err;
};

// Meetings of a workgroup, by slot: the left and right child's summaries
// (com and mass, box, second moments) and the number of arrivals.
template <bool QUAD, int SLOTS>
struct Meet {
    static constexpr int kWords = QUAD ? 16 : 10;
    float v[2][kWords][SLOTS];
    uint32_t cnt[SLOTS];
    __device__ __forceinline__ void put(int side, int k, const LbvhSum &s, const float *Q) {
        const float w[10] = {s.com.x, s.com.y, s.com.z, s.com.w, s.mn.x, s.mn.y, s.mn.z, s.mx.x, s.mx.y, s.mx.z};
#pragma unroll
        for (int i = 0; i < 10; ++i) v[side][i][k] = w[i];
        if constexpr (QUAD) {
#pragma unroll
            for (int i = 0; i < 6; ++i) v[side][10 + i][k] = Q[i];
        }
    }
    __device__ __forceinline__ LbvhSum get(int side, int k, float *Q) const {
        LbvhSum s;
        s.com = make_float4(v[side][0][k], v[side][1][k], v[side][2][k], v[side][3][k]);
        s.mn = make_float4(v[side][4][k], v[side][5][k], v[side][6][k], 0.0f);
        s.mx = make_float4(v[side][7][k], v[side][8][k], v[side][9][k], 0.0f);
        if constexpr (QUAD) {
#pragma unroll
            for (int i = 0; i < 6; ++i) Q[i] = v[side][10 + i][k];
        }
        return s;
    }
};

// A workgroup's finished nodes, whose opening thresholds (which no parent
// needs) are computed in parallel at the end of the pass, and the number of
// nodes it queued.
template <int CAP>
struct PassEnd {
    int id[CAP];
    uint32_t n, queued;
    __device__ __forceinline__ bool add(int node) {
        const uint32_t k = atomicAdd(&n, 1u);
        if (k < (uint32_t)CAP) id[k] = node;
        return k < (uint32_t)CAP;
    }
    __device__ __forceinline__ void finish(const SummPass &P) const {
        __syncthreads();
        const uint32_t m = n < (uint32_t)CAP ? n : (uint32_t)CAP;
        if (P.qout && threadIdx.x == 0) P.qout_n[blockIdx.x] = queued;
        // boxes stored by any thread of the workgroup
        for (uint32_t j = threadIdx.x; j < m; j += blockDim.x)
            P.nodes[id[j]].mac = mac_record(P.bmin[id[j]], P.bmax[id[j]], P.ms.at(P.nodes[id[j]].topo.x));
    }
};

// Climbs from `node` (topology t, summary v and Q, stored) while the parent
// stays in [lo, hi) and this arrival is its second.  slot(p): the meeting
// place of split position p, or -1 to meet in memory.  The parent's topology
// is read a step ahead.
template <bool QUAD, int SLOTS, int CAP, typename Slot>
__device__ __forceinline__ void lbvh_climb(const SummPass &P, int node, int4 t, LbvhSum v, float *Q, int64_t lo,
                                           int64_t hi, Meet<QUAD, SLOTS> &meet, PassEnd<CAP> &end, Slot &&slot) {
    auto topo = [&](int i) { return i >= 0 && i < P.max_nodes ? P.nodes[i].topo : make_int4(-1, -1, -1, -1); };
    int4 tp = topo(t.w);
    while (true) {
        if (!end.add(node)) P.nodes[node].mac = mac_record(v.mn, v.mx, P.ms.at(t.x));
        if (t.w < 0) break;
        const int parent = t.w;
        if (tp.x < 0 || tp.y < 1 || (int64_t)tp.x + tp.y > P.n || tp.z < 0 || (node != tp.z && node != tp.z + 1)) {
            atomicOr(P.err, 4u);
            break;
        }
        if (P.ms.spans(tp)) break;
        if (P.qout && !(tp.x >= lo && (int64_t)tp.x + tp.y <= hi)) {
            P.qout[lo + atomicAdd(&end.queued, 1u)] = (uint32_t)node;  // disjoint subtrees: fewer than the bodies
            break;
        }
        const int4 next = topo(tp.w);
        const int side = node - tp.z;  // 0 left, 1 right
        const int k = slot(side ? t.x - 1 : t.x + t.y - 1);
        LbvhSum o;
        float oq[6];
        if (k >= 0) {
            meet.put(side, k, v, Q);
            if (__hip_atomic_fetch_add(&meet.cnt[k], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) break;
            o = meet.get(1 - side, k, oq);
        } else {
            if (__hip_atomic_fetch_add(&P.flags[parent], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) break;
            const int sib = tp.z + 1 - side;
            o.com = P.nodes[sib].com;
            o.mn = P.bmin[sib];
            o.mx = P.bmax[sib];
            if constexpr (QUAD) {
                const float4 q0 = P.quad[2 * (int64_t)sib], q1 = P.quad[2 * (int64_t)sib + 1];
                oq[0] = q0.x; oq[1] = q0.y; oq[2] = q0.z; oq[3] = q0.w; oq[4] = q1.x; oq[5] = q1.y;
            }
        }
        const LbvhSum l = side ? o : v, r = side ? v : o;
        v = summarize_pair(l, r);
        store_sum(parent, v, P.nodes, P.bmin, P.bmax);
        if constexpr (QUAD) {
            float ql[6], qr[6];
#pragma unroll
            for (int e = 0; e < 6; ++e) {
                ql[e] = side ? oq[e] : Q[e];
                qr[e] = side ? Q[e] : oq[e];
            }
            quad_pair(v.com, l.com, ql, r.com, qr, Q);
            quad_store(P.quad, parent, Q);
        }
        node = parent;
        t = tp;
        tp = next;
    }
}

template <bool QUAD>
__global__ __launch_bounds__(kSummBodies) void k_summ_local(const float4 *__restrict__ bodies,
                                                            const int32_t *__restrict__ leaf_start, SummPass P) {
    __shared__ Meet<QUAD, kSummBodies> meet;
    __shared__ PassEnd<2 * kSummBodies> end;
    meet.cnt[threadIdx.x] = 0;
    if (threadIdx.x == 0) end.n = end.queued = 0;
    __syncthreads();
    const int64_t lo = (int64_t)blockIdx.x * kSummBodies, hi = lo + kSummBodies;
    const int64_t i = lo + threadIdx.x;
    const int s = i < P.n ? leaf_start[i] : -1;
    if (s >= 0) {
        int4 t = make_int4(-1, -1, -1, -1);
        if (s < P.max_nodes) t = P.nodes[s].topo;
        if (t.x != (int)i || t.y < 1 || (int64_t)t.x + t.y > P.n || t.z >= 0) {
            atomicOr(P.err, 4u);
        } else {
            const LbvhSum v = summarize_leaf(t, bodies);
            store_sum(s, v, P.nodes, P.bmin, P.bmax);
            float Q[6];
            if constexpr (QUAD) {
                quad_bodies(bodies, t.x, t.y, v.com.x, v.com.y, v.com.z, Q);
                quad_store(P.quad, s, Q);
            }
            // a parent inside the range splits at a position inside it
            lbvh_climb<QUAD>(P, s, t, v, Q, lo, hi, meet, end,
                             [&](int p) { return (int)(p - lo) & (kSummBodies - 1); });
        }
    }
    end.finish(P);
}

// A later pass: workgroup g owns the `range` bodies from g * range and the
// nodes that the workgroups of the pass before, of `from` bodies each, queued
// there (the parents that stay inside get all their arrivals from it).  Up to
// kSummMeet nodes of a workgroup meet in a hash table of their split
// positions (fewer meetings than nodes), more in memory.
constexpr int kSummMeet = 1024;
constexpr int kSummJoin = 64;  // workgroups of the pass before that one may join

template <bool QUAD>
__global__ __launch_bounds__(1024) void k_summ_queue(const uint32_t *__restrict__ qin, const uint32_t *__restrict__ qin_n,
                                                     int64_t from, int64_t range, SummPass P) {
    __shared__ Meet<QUAD, kSummMeet> meet;
    __shared__ PassEnd<kSummMeet> end;
    __shared__ int key[kSummMeet];
    __shared__ uint32_t before[kSummJoin + 1];
    const int64_t lo = (int64_t)blockIdx.x * range, hi = lo + range;
    for (int i = threadIdx.x; i < kSummMeet; i += blockDim.x) {
        meet.cnt[i] = 0;
        key[i] = -1;
    }
    if (threadIdx.x == 0) end.n = end.queued = 0;
    if (threadIdx.x < kSummJoin) {
        const int64_t g = lo / from + threadIdx.x;
        const uint32_t c = g * from < P.n && g * from < hi ? qin_n[g] : 0u;
        const uint32_t inc = wave_incl_scan(c < (uint32_t)from ? c : (uint32_t)from);
        before[threadIdx.x + 1] = inc;
        if (threadIdx.x == 0) before[0] = 0;
    }
    __syncthreads();
    const uint32_t total = before[kSummJoin];
    const bool in_lds = total <= (uint32_t)kSummMeet;
    for (uint32_t j = threadIdx.x; j < total; j += blockDim.x) {
        int g = 0;  // before[g] <= j < before[g + 1]
#pragma unroll
        for (int o = kSummJoin / 2; o > 0; o >>= 1)
            if (before[g + o] <= j) g += o;
        const int node = (int)qin[(lo / from + g) * from + (j - before[g])];
        if (node < 0 || node >= P.max_nodes) { atomicOr(P.err, 4u); continue; }
        const int4 t = P.nodes[node].topo;
        LbvhSum v;
        v.com = P.nodes[node].com;
        v.mn = P.bmin[node];
        v.mx = P.bmax[node];
        float Q[6];
        if constexpr (QUAD) {
            const float4 q0 = P.quad[2 * (int64_t)node], q1 = P.quad[2 * (int64_t)node + 1];
            Q[0] = q0.x; Q[1] = q0.y; Q[2] = q0.z; Q[3] = q0.w; Q[4] = q1.x; Q[5] = q1.y;
        }
        lbvh_climb<QUAD>(P, node, t, v, Q, lo, hi, meet, end, [&](int p) {
            if (!in_lds) return -1;
            uint32_t h = ((uint32_t)p * 2654435761u) >> 22;  // 10 bits
            for (int probe = 0; probe < kSummMeet; ++probe) {
                const int old = atomicCAS(&key[h], -1, p);
                if (old == -1 || old == p) return (int)h;
                h = (h + 1) & (kSummMeet - 1);
            }
            atomicOr(P.err, 4u);  // unreachable: fewer meetings than nodes
            return 0;
        });
    }
    end.finish(P);
}

template <bool QUAD>
static void launch_summaries(const float4 *bodies, const int32_t *leaf_start, uint32_t *glist, SummPass P, hipStream_t s) {
    // two queues in turn: nodes by body position, then the counts of the workgroups
    uint32_t *q[2] = {glist, glist + 2 * P.n + 64};
    P.qout = q[0];
    P.qout_n = q[0] + P.n;
    hipLaunchKernelGGL(k_summ_local<QUAD>, dim3((unsigned)((P.n + kSummBodies - 1) / kSummBodies)), dim3(kSummBodies), 0,
                       s, bodies, leaf_start, P);
    int64_t from = kSummBodies;
    for (int pass = 0;; ++pass) {
        const uint32_t *in = q[pass & 1], *in_n = q[pass & 1] + P.n;
        const bool last = (P.n + from - 1) / from <= kSummJoin;
        const int64_t range = last ? from * kSummJoin : from * 32;
        P.qout = last ? nullptr : q[(pass + 1) & 1];
        P.qout_n = q[(pass + 1) & 1] + P.n;
        const unsigned g = last ? 1u : (unsigned)((P.n + range - 1) / range);
        hipLaunchKernelGGL(k_summ_queue<QUAD>, dim3(g), dim3(1024), 0, s, in, in_n, from, range, P);
        if (last) break;
        from = range;
    }
}

void launch_lbvh_summaries(const float4 *bodies, int64_t n, NodeRec *nodes, const int32_t *leaf_start,
                           int64_t max_nodes, uint32_t *flags, uint32_t *glist, float4 *bmin, float4 *bmax,
                           float theta, uint32_t *err, hipStream_t s, const MacParam *mp_tab,
                           const uint64_t *keys, int sys_shift, float4 *quad) {
    if (n <= 0) return;
    SummPass P{};
    P.nodes = nodes;
    P.bmin = bmin; P.bmax = bmax; P.quad = quad;
    P.n = n;
    P.max_nodes = max_nodes;
    P.flags = flags;
    mac_threshold(theta, &P.ms.one.mid, &P.ms.one.tie);
    P.ms.tab = mp_tab;
    P.ms.keys = keys;
    P.ms.shift = sys_shift;
    P.err = err;
    if (quad) launch_summaries<true>(bodies, leaf_start, glist, P, s);
    else launch_summaries<false>(bodies, leaf_start, glist, P, s);
}

// ------------------------------------------------------------------ forest
// Independent systems s = 0..S-1 own the ranges [sys_first[s], sys_first[s+1])
// of the concatenated state.  Each gets its own bounding box and 30-bit Morton
// codes over its own bounding cube; the system index sits above the code
// (key = s << 30 | code), so one sort orders every system and, with nodes
// that span systems always split, the radix tree over the concatenation holds
// each system's reference tree as the subtree whose range is that system.

// Boxes of the systems, a workgroup per kSegPart bodies or less of one: the
// workgroups of system i are those from sys_first[i] / kSegPart + i on, of
// which some stay empty.  A system of several parts leaves their boxes in
// `part` (24 bytes for every kSegPart / 4 positions: parts start at least
// kSegPart / 2 apart) for k_seg_fold.  With one workgroup a system 128
// members of 256 to 65,536 bodies took 72 us and one of 239,000 took 229; so
// the former take 16, and 5 to fold.
constexpr int kSegPart = 8192;

__device__ __forceinline__ void seg_reduce(float (&mn)[3], float (&mx)[3]) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            mn[d] = fmin_ref(mn[d], __shfl_xor(mn[d], o, kWave));
            mx[d] = fmax_ref(mx[d], __shfl_xor(mx[d], o, kWave));
        }
}
__device__ __forceinline__ int64_t seg_parts(int64_t n) { return (n + kSegPart - 1) / kSegPart; }
// First position of part j in a system of n bodies: every part of several has
// kSegPart / 2 bodies or more.
__device__ __forceinline__ int64_t seg_start(int64_t n, int64_t parts, int64_t j) { return n * j / parts; }

__global__ __launch_bounds__(256) void k_seg_bbox(const float *__restrict__ x, const float *__restrict__ y,
                                                  const float *__restrict__ z, int nsys,
                                                  const int64_t *__restrict__ sys_first, float *bbox6, float *part) {
    const int64_t block = blockIdx.x;
    int sys = 0, end = nsys;
    while (end - sys > 1) {
        const int mid = (sys + end) >> 1;
        if (sys_first[mid] / kSegPart + mid <= block) sys = mid;
        else end = mid;
    }
    const int64_t first = sys_first[sys], last = sys_first[sys + 1];
    const int64_t n = last - first, parts = n > 0 ? seg_parts(n) : 1, j = block - (first / kSegPart + sys);
    if (j >= parts) return;  // the whole workgroup
    const int64_t lo = first + seg_start(n, parts, j), hi = first + seg_start(n, parts, j + 1);
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        float v[3] = {x[i], y[i], z[i]};
#pragma unroll
        for (int d = 0; d < 3; ++d) { mn[d] = fmin_ref(mn[d], v[d]); mx[d] = fmax_ref(mx[d], v[d]); }
    }
    seg_reduce(mn, mx);
    __shared__ float s_part[4][6];
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0)
        for (int d = 0; d < 3; ++d) { s_part[w][d] = mn[d]; s_part[w][3 + d] = mx[d]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        float r[6];
        for (int d = 0; d < 6; ++d) r[d] = s_part[0][d];
        for (int ww = 1; ww < 4; ++ww)
            for (int d = 0; d < 3; ++d) { r[d] = fmin_ref(r[d], s_part[ww][d]); r[3 + d] = fmax_ref(r[3 + d], s_part[ww][3 + d]); }
        float *const out = parts > 1 ? part + 6 * (lo / (kSegPart / 4)) : bbox6 + 6 * (int64_t)sys;
        for (int d = 0; d < 6; ++d) out[d] = r[d];
    }
}

// The boxes of the systems of several parts, a wave each.
__global__ __launch_bounds__(64) void k_seg_fold(const int64_t *__restrict__ sys_first, const float *__restrict__ part,
                                                 float *bbox6) {
    const int sys = blockIdx.x;
    const int64_t first = sys_first[sys], n = sys_first[sys + 1] - first, parts = seg_parts(n);
    if (parts <= 1) return;
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int64_t j = threadIdx.x; j < parts; j += kWave) {
        const int64_t lo = first + seg_start(n, parts, j);
        const float *const r = part + 6 * (lo / (kSegPart / 4));
#pragma unroll
        for (int d = 0; d < 3; ++d) { mn[d] = fmin_ref(mn[d], r[d]); mx[d] = fmax_ref(mx[d], r[3 + d]); }
    }
    seg_reduce(mn, mx);
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d) { bbox6[6 * (int64_t)sys + d] = mn[d]; bbox6[6 * (int64_t)sys + 3 + d] = mx[d]; }
}

__global__ __launch_bounds__(256) void k_forest_keys(const float *__restrict__ x, const float *__restrict__ y,
                                                     const float *__restrict__ z, int64_t n,
                                                     const uint32_t *__restrict__ bsys,
                                                     const float *__restrict__ bbox6, uint64_t *__restrict__ keys,
                                                     uint32_t *__restrict__ idx, uint32_t *__restrict__ ghist,
                                                     int passes, int shift) {
    __shared__ uint32_t h[8 * kRadix];
    const DigitCount dc{h, passes, shift};
    dc.clear();
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t sys = bsys[i];
        const uint64_t k = ((uint64_t)sys << 30) | (uint64_t)morton_key<uint32_t>(x[i], y[i], z[i], bbox6 + 6 * sys);
        keys[i] = k;
        idx[i] = (uint32_t)i;
        dc.add(k);
    }
    __syncthreads();
    dc.store(ghist);
}

// A node is the root of system s iff its range lies inside s and its
// parent's range does not.
__global__ __launch_bounds__(256) void k_forest_roots(const NodeRec *__restrict__ nodes,
                                                      const uint32_t *__restrict__ node_count, int64_t max_nodes,
                                                      const uint64_t *__restrict__ keys, int64_t n, int nsys,
                                                      int32_t *sys_root, uint32_t *err) {
    const int64_t slot = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (slot >= *node_count || slot >= max_nodes) return;
    const int4 t = nodes[slot].topo;
    if (t.x < 0 || t.y < 1 || (int64_t)t.x + t.y > n) { atomicOr(err, 4u); return; }
    const uint64_t s0 = keys[t.x] >> 30, s1 = keys[t.x + t.y - 1] >> 30;
    if (s0 != s1) return;
    if (t.w >= 0) {
        if ((int64_t)t.w >= max_nodes) { atomicOr(err, 4u); return; }
        const int4 tp = nodes[t.w].topo;
        if (tp.x < 0 || tp.y < 1 || (int64_t)tp.x + tp.y > n) { atomicOr(err, 4u); return; }
        if ((keys[tp.x] >> 30) == (keys[tp.x + tp.y - 1] >> 30)) return;
    }
    if (s0 < (uint64_t)nsys) sys_root[s0] = (int32_t)slot;
}

void launch_forest_build(const float *x, const float *y, const float *z, int64_t n, int nsys,
                         const int64_t *sys_first, int64_t largest, const uint32_t *bsys, float *bbox6,
                         uint64_t *keys, uint32_t *idx,
                         uint64_t *keys_alt, uint32_t *idx_alt, uint32_t *sort_status, FillSet &fills, uint32_t *err,
                         hipStream_t s) {
    if (n <= 0 || nsys <= 0) return;
    int sbits = 0;
    while ((1ll << sbits) < nsys) ++sbits;
    const SortPlan plan = sort_plan(n, 30 + sbits, false);
    fills.add(sort_status, sort_clear_words(n, plan));
    launch_seg_bbox(x, y, z, n, nsys, sys_first, largest, bbox6, (float *)keys, s);
    launch_fills(fills, s);
    int64_t blocks = (n + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_forest_keys, dim3((unsigned)blocks), dim3(256), 0, s, x, y, z, n, bsys, bbox6,
                       plan.from_alt ? keys_alt : keys, plan.from_alt ? idx_alt : idx, sort_status, plan.passes,
                       plan.shift);
    launch_sort(keys, idx, keys_alt, idx_alt, n, 64, plan, sort_status, err, s);
}

void launch_seg_bbox(const float *x, const float *y, const float *z, int64_t n, int nsys, const int64_t *sys_first,
                     int64_t largest, float *bbox6, float *part, hipStream_t s) {
    if (nsys <= 0) return;
    hipLaunchKernelGGL(k_seg_bbox, dim3((unsigned)(n / kSegPart + nsys)), dim3(256), 0, s, x, y, z, nsys, sys_first,
                       bbox6, part);
    if (largest > kSegPart) hipLaunchKernelGGL(k_seg_fold, dim3((unsigned)nsys), dim3(64), 0, s, sys_first, part, bbox6);
}

void launch_forest_roots(const NodeRec *nodes, const uint32_t *node_count, int64_t max_nodes, const uint64_t *keys,
                         int64_t n, int nsys, int32_t *sys_root, uint32_t *err, hipStream_t s) {
    if (n <= 0 || nsys <= 0) return;
    launch_fill_u32((uint32_t *)sys_root, 0xFFFFFFFFu, nsys, s);
    hipLaunchKernelGGL(k_forest_roots, dim3((unsigned)((max_nodes + 255) / 256)), dim3(256), 0, s, nodes, node_count,
                       max_nodes, keys, n, nsys, sys_root, err);
}

}  // namespace nbg
