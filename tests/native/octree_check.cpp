// A whole octree pass on the CPU, every buffer exactly as large as the
// library makes it: box, keys, sort, topology, gather, summaries and the walk.
//   octree_check FILE N LEAF DEPTH THETA EPS2 OUT FROM TO ORDERED
// FILE: x, y, z, m (N floats each); OUT: the accelerations of the walk's
// targets FROM .. TO - 1 by body (others 0), and the interaction counts.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../n-body_amd/csrc/launch.hpp"

using namespace nbg;

template <typename T>
static void alloc(T **p, int64_t n) {
    *p = (T *)std::malloc((size_t)n * sizeof(T));
    for (size_t i = 0; i < (size_t)n * sizeof(T); ++i) ((unsigned char *)*p)[i] = 0xA5;
}

int main(int argc, char **argv) {
    if (argc != 11) return 2;
    const int64_t n = std::atoll(argv[2]), from = std::atoll(argv[8]), to = std::atoll(argv[9]);
    const int leaf = std::atoi(argv[3]), depth = std::atoi(argv[4]);
    const float theta = (float)std::atof(argv[5]), eps2 = (float)std::atof(argv[6]);
    float *c[4];
    FILE *f = std::fopen(argv[1], "rb");
    if (!f) return 2;
    for (auto &v : c) {
        alloc(&v, n);
        if (std::fread(v, 4, n, f) != (size_t)n) return 2;
    }
    std::fclose(f);
    const int64_t cap = octree_capacity(n, leaf, depth);
    OctBuffers b;
    alloc(&b.key_hi, n); alloc(&b.key_lo, n); alloc(&b.lo_sorted, n);
    alloc(&b.nown, n); alloc(&b.nbase, n);
    alloc(&b.nfirst, cap); alloc(&b.ncount, cap); alloc(&b.nparent, cap); alloc(&b.nmeta, cap);
    alloc(&b.occ, cap); alloc(&b.cb, cap); alloc(&b.flags, cap); alloc(&b.glist, 2 * oct_queue_words(n));
    alloc(&b.scan_ws, oct_scan_words(n, cap));
    alloc(&b.nodes, cap); alloc(&b.centre, cap); alloc(&b.thr, 64); alloc(&b.misc, 64);
    b.cap = cap;
    b.n = n;
    uint64_t *keys, *keys_alt;
    uint32_t *idx, *idx_alt, *status;
    int32_t *leaf_start;
    float4 *bodies;
    float *partials, bbox[6], *a[3];
    alloc(&keys, n); alloc(&keys_alt, n); alloc(&idx, n); alloc(&idx_alt, n); alloc(&leaf_start, n); alloc(&bodies, n);
    alloc(&status, sort_status_words(n, 63));
    alloc(&partials, 6 * kBBoxBlocks);
    for (auto &v : a) {
        alloc(&v, n);
        for (int64_t i = 0; i < n; ++i) v[i] = 0.0f;
    }
    uint32_t err = 0;
    unsigned long long counts[6] = {};

    const bool lo = oct_has_lo(depth);
    const SortPlan plan = sort_plan(n, 63, lo);
    FillSet fills;
    fills.add(status, sort_clear_words(n, plan));
    oct_fills(fills, b, n, leaf_start);
    auto say = [](const char *what) { std::printf("%s\n", what); std::fflush(stdout); };
    const int parts = launch_bbox(c[0], c[1], c[2], n, partials, fills, nullptr);
    say("keys");
    launch_octree_keys(c[0], c[1], c[2], n, partials, parts, bbox, depth, theta, plan, b, keys, idx_alt, keys_alt, idx,
                       status, nullptr);
    say("sort");
    launch_sort(keys, idx_alt, keys_alt, idx, n, 63, plan, status, &err, nullptr, lo ? b.key_lo : nullptr, b.lo_sorted);
    say("topology");
    launch_octree_topology(n, bbox, leaf, depth, b, keys, idx_alt, idx, leaf_start, &err, nullptr);
    launch_gather(c[0], c[1], c[2], c[3], idx, n, bodies, nullptr);
    say("summaries");
    launch_octree_summaries(bodies, n, b, leaf_start, &err, nullptr);
    std::printf("nodes %u of %lld, err %u\n", b.misc[0], (long long)cap, err);
    say("walk");
    WalkArgs w{};
    w.n = n;
    w.bodies = bodies;
    w.nt = to - from;
    w.targets = bodies + from;
    std::vector<uint32_t> perm(to - from);
    for (int64_t i = from; i < to; ++i) perm[i - from] = (uint32_t)(i - from);
    w.perm = perm.data();
    w.onodes = b.nodes;
    w.levels = depth + 2;
    w.theta = theta;
    w.G = 1.0f;
    w.eps2 = eps2;
    w.max_nodes = cap;
    w.ax = a[0]; w.ay = a[1]; w.az = a[2];
    w.counts = counts;
    w.err = &err;
    const int ordered = std::atoi(argv[10]);
    w.split = ordered ? ordered_split_waves((n + 63) / 64, true, n) : fast_split_waves((n + 63) / 64);
    launch_walk_oct(w, ordered, 1, nullptr);
    std::printf("err %u pp %llu np %llu\n", err, counts[0], counts[1]);
    f = std::fopen(argv[7], "wb");
    std::vector<float> out(3 * n, 0.0f);
    for (int64_t i = from; i < to; ++i)
        for (int d = 0; d < 3; ++d) out[3 * (size_t)idx[i] + d] = a[d][i - from];
    std::fwrite(out.data(), 4, out.size(), f);
    std::fclose(f);
    return err != 0;
}
