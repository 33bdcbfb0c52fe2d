// The last stage of the build's sort (build.hip) on the CPU.
//   failed: indices as a radix pass leaves them that gave up its look-back
//     (some never written): an error is reported, nothing is read out of bounds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../../n-body_amd/csrc/launch.hpp"

using namespace nbg;

static int failed() {
    int bad = 0;
    for (int n : {50, 700, 3000})
        for (int lo = 0; lo < 2; ++lo) {
            // no radix pass: the last stage alone, from the _alt buffers
            const SortPlan plan{0, 31, true, true};
            std::vector<uint64_t> keys(n), alt(n);
            std::vector<uint32_t> idx(n), idx_alt(n), status((size_t)sort_status_words(n, 64), 0u);
            uint64_t *low = (uint64_t *)std::malloc(n * sizeof(uint64_t)), *low_out = (uint64_t *)std::malloc(n * sizeof(uint64_t));
            std::mt19937 g(n);
            for (int i = 0; i < n; ++i) {
                alt[i] = n == 50 ? i / 4 : g() & 3u;  // one run, many equal keys
                idx_alt[i] = (uint32_t)(i % 5 != 1 ? i : n + 1);
                low[i] = g();
            }
            uint32_t err = 0;
            std::printf("failed n=%d lo=%d\n", n, lo);
            std::fflush(stdout);
            launch_sort(keys.data(), idx.data(), alt.data(), idx_alt.data(), n, 63, plan, status.data(), &err, nullptr,
                        lo ? low : nullptr, lo ? low_out : nullptr);
            if (!(err & 1u)) ++bad;
            std::free(low);
            std::free(low_out);
        }
    return bad;
}

int main(int argc, char **argv) {
    int bad = 0;
    if (argc > 1 && !std::strcmp(argv[1], "failed")) bad = failed();
    if (bad) std::printf("%d wrong\n", bad);
    return bad != 0;
}
