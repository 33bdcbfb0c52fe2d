// The work of one group of 64 targets, shared by the Barnes-Hut walks.
#pragma once

#include "device.hpp"
#include "launch.hpp"

namespace nbg {

// The forest's order of workgroups: runs of kTurn consecutive ones (2,048
// targets of the FAST walks) on one XCD, the XCDs in turn.  A single system
// gives each XCD one eighth of itself; members differ in their cost per body
// (a lower angle, a larger tree), and an eighth of a forest can be most of its
// work.  A FAST pass, ms: eight members of 200,000 bodies at theta 0.3, 0.5
// and 0.7 21.9 -> 7.0, 128 of 256 to 65,536 bodies 5.7 -> 5.3, such octrees
// sorted by size 3.7 -> 3.5.  Which of eight runs an XCD takes moves on by an
// irrational step (the fraction of the root of 2, in eighths), so that members
// of 16,384 bodies, eight runs each, do not leave their dense eighths to one
// XCD: 256 of them at leaf 16 16.9 -> 12.7 ms, octrees at leaf 64 14.4 -> 12.2.
constexpr unsigned kTurn = 32;
__device__ __forceinline__ unsigned xcd_turns(unsigned b, unsigned blocks) {
    const unsigned whole = blocks / (8 * kTurn) * (8 * kTurn);
    if (b >= whole) return b;
    const unsigned xcd = b % 8, k = b / 8;  // the k-th workgroup of its XCD
    const unsigned q = k / kTurn;          // its q-th run, of eight that follow each other
    return (q * 8 + (xcd + (q * 0x6A09E667u >> 29)) % 8) * kTurn + k % kTurn;
}

// The workgroup's place in the walk's order.
template <bool FOREST>
__device__ __forceinline__ unsigned walk_block() {
    return FOREST ? xcd_turns(blockIdx.x, gridDim.x) : (unsigned)xcd_block(blockIdx.x, gridDim.x);
}

// The targets, root and rule of group w: the whole tree for one system, or
// the system that owns group w in a forest (all wave-uniform).
struct WaveTask {
    int64_t base, end;
    int root;
    float G, eps2;
};

template <bool FOREST>
__device__ __forceinline__ WaveTask wave_task(const WalkArgs &a, int64_t w) {
    WaveTask t;
    if (!FOREST) {
        t.base = w * kWave; t.end = a.nt; t.root = 0; t.G = a.G; t.eps2 = a.eps2;
        return t;
    }
    if (w >= a.nwaves) {
        t.base = 0; t.end = 0; t.root = 0; t.G = a.G; t.eps2 = a.eps2;
        return t;
    }
    int lo = 0, hi = a.nsys;  // wave_first[lo] <= w < wave_first[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (a.wave_first[mid] <= w) lo = mid;
        else hi = mid;
    }
    t.base = a.sys_first[lo] + (w - a.wave_first[lo]) * kWave;
    t.end = a.sys_first[lo + 1];
    t.root = a.sys_root[lo];
    const float4 q = a.sys_prm[lo];
    t.G = q.x;
    t.eps2 = q.y;
    return t;
}

}  // namespace nbg
