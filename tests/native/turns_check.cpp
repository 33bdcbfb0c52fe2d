// The forest's order of workgroups: every workgroup once, and where the
// members are alike no XCD gets the same part of each of them.
#include "simt.hpp"

#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../n-body_amd/csrc/walk_task.hpp"

int main() {
    for (unsigned member : {8u, 64u, 128u, 256u, 300u, 512u, 1024u, 2048u, 4096u, 8192u}) {
        for (unsigned members : {1u, 3u, 64u, 1000u}) {
            const unsigned blocks = member * members;
            std::vector<char> seen(blocks, 0);
            std::vector<unsigned> part(8 * 8, 0);  // workgroups of a member's eighth on an XCD
            for (unsigned b = 0; b < blocks; ++b) {
                const unsigned w = nbg::xcd_turns(b, blocks);
                if (w >= blocks || seen[w]) {
                    std::printf("%u members of %u: workgroup %u taken by %u too\n", members, member, w, b);
                    return 1;
                }
                seen[w] = 1;
                ++part[b % 8 * 8 + std::min(w % member / (member / 8), 7u)];
            }
            std::printf("%u %u %.3f\n", members, member, *std::max_element(part.begin(), part.end()) / (blocks / 64.0));
        }
    }
    return 0;
}
