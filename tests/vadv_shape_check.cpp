// Host-side check of the launch rules of the register-column vadv
// (stencil_benchmarks_amd/csrc/vadv_regs.h, sb_internal.h).  Exits non-zero on
// the first rule that does not hold.
#include <cstdio>
#include <vector>

#include "../stencil_benchmarks_amd/csrc/sb_internal.h"
#include "../stencil_benchmarks_amd/csrc/vadv_regs.h"

// Every workgroup takes an item of its own, whatever the run length.
static int check_remap() {
    for (uint32_t xcds : {1u, 2u, 8u})
        for (uint32_t total : {1u, 7u, 8u, 9u, 64u, 127u, 128u, 129u, 256u, 1000u, 2500u, 2048u})
            for (uint32_t chunk : {1u, 3u, 16u, total / xcds, total}) {
                if (chunk == 0) continue;
                std::vector<char> seen(total, 0);
                for (uint32_t b = 0; b < total; ++b) {
                    const uint32_t n = sb::xcd_chunk_remap(b, total, xcds, chunk);
                    if (n >= total || seen[n]++) {
                        std::printf("workgroup %u of %u, %u XCDs, runs of %u: item %u\n", b, total, xcds,
                                    chunk, n);
                        return 1;
                    }
                }
            }
    return 0;
}

int main() {
    if (check_remap()) return 1;
    std::printf("ok\n");
    return 0;
}
