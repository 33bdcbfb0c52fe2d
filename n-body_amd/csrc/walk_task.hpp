// The work of one group of 64 targets, shared by the Barnes-Hut walks.
#pragma once

#include "device.hpp"
#include "launch.hpp"

namespace nbg {

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
