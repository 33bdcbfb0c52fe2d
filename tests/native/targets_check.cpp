// The compact groups of a walk's targets (targets.hip) on the CPU: every body
// of a block, whole or ragged, comes out once, with its place in perm, in the
// same order whatever the order of the waves.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../n-body_amd/csrc/launch.hpp"

using namespace nbg;

int main() {
    int bad = 0;
    for (int n : {1, 15, 1000, 1024, 1025, 5000}) {
        for (int flat = 0; flat < 2; ++flat) {
            std::mt19937 g(n + flat);
            std::normal_distribution<float> d(0.0f, 1.0f);
            std::vector<float4> in(n), out(n);
            std::vector<uint32_t> perm(n), got(n, ~0u);
            for (int i = 0; i < n; ++i) {
                in[i] = make_float4(flat ? 0.5f : d(g), d(g), flat && i % 3 ? 0.0f : d(g), (float)i);
                perm[i] = (uint32_t)(n - 1 - i);
            }
            launch_group_targets(in.data(), perm.data(), n, out.data(), got.data(), nullptr);
            uint64_t hash = 1469598103934665603ull;
            for (int b = 0; b < n; b += 1024) {
                const int e = b + 1024 < n ? b + 1024 : n;
                std::vector<int> seen(e - b, 0);
                for (int i = b; i < e; ++i) {
                    const int body = (int)out[i].w;
                    if (body < b || body >= e || seen[body - b]++ || got[i] != perm[body] || out[i].x != in[body].x ||
                        out[i].y != in[body].y || out[i].z != in[body].z)
                        ++bad;
                    hash = (hash ^ (uint64_t)body) * 1099511628211ull;
                }
            }
            std::printf("%d %d %016llx\n", n, flat, (unsigned long long)hash);
        }
    }
    if (bad) {
        std::printf("%d targets are not the block's bodies once each\n", bad);
        return 1;
    }
    return 0;
}
