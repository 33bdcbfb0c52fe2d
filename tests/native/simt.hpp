// Runs HIP kernels on the CPU, for the tests that look for races and reads out
// of bounds: force-included before a .hip file that is compiled as C++.
//
// A workgroup's threads are fibres.  A thread runs until it needs others: a
// cross-lane operation waits for its wave (all of whose live lanes must reach
// the same one; lanes that have returned are left out), __syncthreads for the
// workgroup.  Between barriers the waves run one after the other, in an order
// that NBG_SIMT_ORDER picks (0 ascending, 1 descending, >= 2 shuffled anew at
// every barrier with that seed), so a wave gets as far ahead of the others as
// a barrier lets it.  Workgroups run one after the other.  LDS is filled with
// 0xA5 before each workgroup.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>

#undef __global__
#undef __device__
#undef __host__
#undef __shared__
#undef __launch_bounds__
#undef __forceinline__
#define __global__
#define __device__
#define __host__
#define __launch_bounds__(...)
#define __forceinline__ inline
#ifdef SIMT_REDZONES  // one after the other with AddressSanitizer's red zones between, and not filled
#define __shared__ static
#else
#define __shared__ static __attribute__((section("simt_lds")))
#endif

namespace simt {

struct Fibre {
    dim3 tid, bid, bdim, gdim;
    int lane = 0, wave = 0;
};
extern Fibre *cur;

// Waits until every live lane of the wave is here with its word, and returns
// the wave's words (64); *live: the lanes that take part.
const uint64_t *meet(uint64_t word, uint64_t *live, const char *file, int line);
void barrier();
void launch(dim3 grid, dim3 block, const std::function<void()> &body);

}  // namespace simt

#define threadIdx (simt::cur->tid)
#define blockIdx (simt::cur->bid)
#define blockDim (simt::cur->bdim)
#define gridDim (simt::cur->gdim)
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    simt::launch(grid, block, [=] { kernel(__VA_ARGS__); })

#define SIMT_AT const char *file = __builtin_FILE(), int line = __builtin_LINE()
#define __syncthreads() simt::barrier()

template <typename T>
inline uint64_t simt_word(T v) {
    static_assert(sizeof(T) <= 8, "");
    uint64_t w = 0;
    std::memcpy(&w, &v, sizeof v);
    return w;
}
template <typename T>
inline T simt_from(const uint64_t *w, int lane) {
    T v;
    std::memcpy(&v, &w[lane & 63], sizeof v);
    return v;
}
inline uint64_t __ballot(bool p, SIMT_AT) {
    uint64_t live, b = 0;
    const uint64_t *w = simt::meet(p, &live, file, line);
    for (int i = 0; i < 64; ++i)
        if ((live >> i & 1) && w[i]) b |= 1ull << i;
    return b;
}
template <typename T>
inline T __shfl(T v, int lane, int = 64, SIMT_AT) {
    uint64_t live;
    return simt_from<T>(simt::meet(simt_word(v), &live, file, line), lane);
}
template <typename T>
inline T __shfl_xor(T v, int x, int = 64, SIMT_AT) {
    uint64_t live;
    return simt_from<T>(simt::meet(simt_word(v), &live, file, line), simt::cur->lane ^ x);
}
template <typename T>
inline T __shfl_up(T v, int o, int = 64, SIMT_AT) {
    uint64_t live;
    const int l = simt::cur->lane;
    return simt_from<T>(simt::meet(simt_word(v), &live, file, line), l < o ? l : l - o);
}
template <typename T>
inline T __shfl_down(T v, int o, int = 64, SIMT_AT) {
    uint64_t live;
    const int l = simt::cur->lane;
    return simt_from<T>(simt::meet(simt_word(v), &live, file, line), l + o > 63 ? l : l + o);
}
inline int __builtin_amdgcn_readfirstlane(int v, SIMT_AT) {
    uint64_t live;
    const uint64_t *w = simt::meet(simt_word(v), &live, file, line);
    return simt_from<int>(w, __builtin_ctzll(live));
}
inline int __builtin_amdgcn_readlane(int v, int lane, SIMT_AT) {
    uint64_t live;
    return simt_from<int>(simt::meet(simt_word(v), &live, file, line), lane);
}
inline void __builtin_amdgcn_wave_barrier(SIMT_AT) {
    uint64_t live;
    simt::meet(0, &live, file, line);
}
inline void __builtin_amdgcn_fence(int, const char *scope, SIMT_AT) {
    uint64_t live;
    if (scope[0] == 'w' && scope[1] == 'a') simt::meet(0, &live, file, line);
}
inline void __builtin_amdgcn_s_sleep(int) {}
inline void __builtin_amdgcn_s_waitcnt(int) {}
inline int __builtin_amdgcn_ds_bpermute(int addr, int v, SIMT_AT) {
    uint64_t live;
    return simt_from<int>(simt::meet(simt_word(v), &live, file, line), addr / 4);
}
struct SimtPair {
    uint32_t v[2];
    uint32_t operator[](int i) const { return v[i]; }
};
inline SimtPair __builtin_amdgcn_permlane16_swap(uint32_t a, uint32_t b, bool, bool, SIMT_AT) {
    uint64_t live;
    const uint64_t *w = simt::meet(a | (uint64_t)b << 32, &live, file, line);
    const int l = simt::cur->lane, row = l / 16;
    auto A = [&](int lane) { return (uint32_t)w[lane]; };
    auto B = [&](int lane) { return (uint32_t)(w[lane] >> 32); };
    return row & 1 ? SimtPair{{B(l - 16), b}} : SimtPair{{a, A(l + 16)}};
}
inline SimtPair __builtin_amdgcn_permlane32_swap(uint32_t a, uint32_t b, bool, bool, SIMT_AT) {
    uint64_t live;
    const uint64_t *w = simt::meet(a | (uint64_t)b << 32, &live, file, line);
    const int l = simt::cur->lane;
    return l < 32 ? SimtPair{{a, (uint32_t)w[l + 32]}} : SimtPair{{(uint32_t)(w[l - 32] >> 32), b}};
}
inline int __builtin_amdgcn_mov_dpp(int v, int ctrl, int, int, bool, SIMT_AT) {
    uint64_t live;
    const uint64_t *w = simt::meet(simt_word(v), &live, file, line);
    const int l = simt::cur->lane, row = l & ~15, i = l & 15;
    if (ctrl < 0x100) return simt_from<int>(w, (l & ~3) + (ctrl >> (2 * (l & 3)) & 3));
    if (ctrl > 0x120 && ctrl < 0x130) return simt_from<int>(w, row + ((i - (ctrl & 15)) & 15));
    if (ctrl == 0x140) return simt_from<int>(w, row + (15 - i));
    if (ctrl == 0x141) return simt_from<int>(w, (l & ~7) + (7 - (l & 7)));
    std::abort();
}
// row_shr (0x111 ..), row_bcast:15 and :31; lanes without a source take 0
// (bound) or old, rows not in the mask old
inline int __builtin_amdgcn_update_dpp(int old, int v, int ctrl, int rows, int, bool bound, SIMT_AT) {
    uint64_t live;
    const uint64_t *w = simt::meet(simt_word(v), &live, file, line);
    const int l = simt::cur->lane;
    if (!(rows >> (l / 16) & 1)) return old;
    int from = -1;
    if (ctrl > 0x110 && ctrl < 0x120) from = (l & 15) >= (ctrl & 15) ? l - (ctrl & 15) : -1;
    else if (ctrl == 0x142) from = l >= 16 ? (l & ~15) - 1 : -1;
    else if (ctrl == 0x143) from = l >= 32 ? 31 : -1;
    else std::abort();
    return from >= 0 ? simt_from<int>(w, from) : bound ? 0 : old;
}
inline bool __builtin_amdgcn_inverse_ballot_w64(uint64_t b) { return b >> simt::cur->lane & 1; }
inline uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t m, uint32_t a) {
    const int l = simt::cur->lane;
    return a + (uint32_t)__builtin_popcount(l >= 32 ? m : m & ((1u << l) - 1u));
}
inline uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t m, uint32_t a) {
    const int l = simt::cur->lane;
    return a + (uint32_t)__builtin_popcount(l <= 32 ? 0u : m & ((1u << (l - 32)) - 1u));
}
inline double __builtin_amdgcn_rcp(double d) { return 1.0 / d; }
inline float __builtin_amdgcn_rsqf(float v) { return 1.0f / std::sqrt(v); }
inline int32_t __builtin_amdgcn_sbfe(int32_t v, uint32_t off, uint32_t width) {
    return (int32_t)((uint32_t)v << (32 - off - width)) >> (32 - width);
}
// the one asm of the kernels: v_addc with the lane's bit of b as the carry in
#define asm(...) (carry = 0, v = 2u * v + (uint32_t)(b >> simt::cur->lane & 1))

template <typename T, typename U>
inline T simt_rmw_add(T *p, U v) {
    const T o = *p;
    *p = (T)(o + (T)v);
    return o;
}
inline uint32_t atomicAdd(uint32_t *p, uint32_t v) { return simt_rmw_add(p, v); }
inline int atomicAdd(int *p, int v) { return simt_rmw_add(p, v); }
inline unsigned long long atomicAdd(unsigned long long *p, unsigned long long v) { return simt_rmw_add(p, v); }
inline uint32_t atomicMax(uint32_t *p, uint32_t v) {
    const uint32_t o = *p;
    if (v > o) *p = v;
    return o;
}
inline uint32_t atomicOr(uint32_t *p, uint32_t v) {
    const uint32_t o = *p;
    *p = o | v;
    return o;
}
inline int atomicCAS(int *p, int want, int v) {
    const int o = *p;
    if (o == want) *p = v;
    return o;
}
#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_fetch_add(p, v, order, scope) simt_rmw_add(p, v)
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))
inline void __threadfence_block() {}
inline void __threadfence() {}

inline int __popc(uint32_t v) { return __builtin_popcount(v); }
inline int __popcll(uint64_t v) { return __builtin_popcountll(v); }
inline int __clz(uint32_t v) { return v ? __builtin_clz(v) : 32; }
inline int __clzll(long long v) { return v ? __builtin_clzll((unsigned long long)v) : 64; }
inline float __uint_as_float(uint32_t v) { return __builtin_bit_cast(float, v); }
inline uint32_t __float_as_uint(float v) { return (uint32_t)simt_word(v); }
inline int __float_as_int(float v) { return (int)simt_word(v); }
inline float __int_as_float(int v) { return __uint_as_float((uint32_t)v); }
