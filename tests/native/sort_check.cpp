// The last stage of the build's sort (build.hip) on the CPU.
//   failed: indices as a radix pass leaves them that gave up its look-back
//     (some never written): an error is reported, nothing is read out of bounds.
//   fills: more ranges than a kernel takes are all set.
//   runs: keys that share the sorted bits in runs on both sides of the run
//     lengths at which the stage changes its way: the stable order.
#include <algorithm>
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

static int runs() {
    int bad = 0;
    // lengths of the runs, one after the other, until n keys are there
    const std::vector<std::vector<int>> shapes = {{256, 257, 1, 3}, {4096, 1, 300}, {4097, 2}, {9000}, {300}, {5, 20000, 700}, {16384, 9}, {16385, 9}};
    for (size_t q = 0; q < shapes.size(); ++q)
        for (int lo = 0; lo < 2; ++lo) {
            const int n = 12345 + 8191 * (int)(q % 3);
            const SortPlan plan{0, 31, true, true};
            std::vector<uint64_t> keys(n), alt(n), low(n), low_out(n);
            std::vector<uint32_t> idx(n), idx_alt(n), status((size_t)sort_status_words(n, 64), 0xA5A5A5A5u);
            std::fill(status.begin(), status.begin() + sort_clear_words(n, plan), 0u);
            std::mt19937_64 g(q);
            uint64_t prefix = 0;
            for (int i = 0, r = 0; i < n; ++prefix, ++r)
                for (int k = shapes[q][r % shapes[q].size()]; k > 0 && i < n; --k, ++i)
                    alt[i] = prefix << 31 | (g() & (g() % 7 ? 0x7FFFFFFFull : 0x3ull));
            // equal prefixes stand in the order of the index
            std::vector<uint32_t> at(n);
            for (int i = 0; i < n; ++i) at[i] = (uint32_t)i;
            std::shuffle(at.begin(), at.end(), g);
            for (int i = 0; i < n;) {
                int e = i;
                while (e < n && alt[e] >> 31 == alt[i] >> 31) ++e;
                std::sort(at.begin() + i, at.begin() + e);
                i = e;
            }
            for (int i = 0; i < n; ++i) {
                idx_alt[i] = at[i];
                low[at[i]] = lo ? g() & (g() % 3 ? 0x7FFFFFFFFFull : 0x7ull) : 0;
            }
            struct E { uint64_t k, l; uint32_t v; };
            std::vector<E> want(n);
            for (int i = 0; i < n; ++i) want[i] = E{alt[i], low[at[i]], at[i]};
            std::sort(want.begin(), want.end(), [](const E &a, const E &b) {
                return a.k != b.k ? a.k < b.k : a.l != b.l ? a.l < b.l : a.v < b.v;
            });
            uint32_t err = 0;
            launch_sort(keys.data(), idx.data(), alt.data(), idx_alt.data(), n, 63, plan, status.data(), &err, nullptr,
                        lo ? low.data() : nullptr, lo ? low_out.data() : nullptr);
            int wrong = err != 0;
            for (int i = 0; i < n; ++i)
                wrong += keys[i] != want[i].k || idx[i] != want[i].v || (lo && low_out[i] != want[i].l);
            std::printf("runs %zu lo=%d n=%d wrong %d\n", q, lo, n, wrong);
            bad += wrong != 0;
        }
    return bad;
}

static int fills() {
    int bad = 0;
    for (int box = 0; box < 2; ++box)
        for (int count : {1, 10, 11, 25}) {
            std::vector<std::vector<uint32_t>> mem(count);
            FillSet f;
            for (int i = 0; i < count; ++i) {
                mem[i].assign(3 + 500 * (i % 3), 0xA5A5A5A5u);
                f.add(mem[i].data(), (int64_t)mem[i].size(), (uint32_t)i);
            }
            std::vector<float> x(100, 1.0f), partials(6 * kBBoxBlocks);
            if (box) launch_bbox(x.data(), x.data(), x.data(), 100, partials.data(), f, nullptr);
            else launch_fills(f, nullptr);
            int wrong = 0;
            for (int i = 0; i < count; ++i)
                for (uint32_t v : mem[i]) wrong += v != (uint32_t)i;
            std::printf("fills box=%d count=%d wrong %d\n", box, count, wrong);
            bad += wrong != 0;
        }
    return bad;
}

int main(int argc, char **argv) {
    int bad = 0;
    if (argc > 1 && !std::strcmp(argv[1], "failed")) bad = failed();
    if (argc > 1 && !std::strcmp(argv[1], "fills")) bad = fills();
    if (argc > 1 && !std::strcmp(argv[1], "runs")) bad = runs();
    if (bad) std::printf("%d wrong\n", bad);
    return bad != 0;
}
