// Host check of the tile order over the XCDs (mr-lbm_amd/csrc/kernels.h): the
// regrouped order is a permutation that keeps the last n % 256 positions, and
// workgroups of one XCD (b % 8) take runs of 32 consecutive positions; beyond
// the byte limit nothing moves. Prints "ok" and exits 0 on success.
#include <cstdio>
#include <vector>

#include "../mr-lbm_amd/csrc/kernels.h"

using namespace mrlbm;

int main() {
    int failures = 0;
    for (size_t n : {0, 1, 8, 31, 255, 256, 257, 511, 512, 540, 1000, 4096, 32768, 100001}) {
        if (xcd_group_end(n, XCD_GROUP_MAX_BYTES) != 0) failures++;
        const uint32_t end = xcd_group_end(n, 1.0);
        if (end > n || n - end >= 256 || end % 256) failures++;
        std::vector<int> seen(n, 0);
        for (uint32_t b = 0; b < n; b++) {
            const uint32_t t = xcd_grouped(b, end);
            if (t >= n) {
                failures++;
                continue;
            }
            seen[t]++;
            if (b >= end ? t != b : (t / 32 % 8 != b % 8 || t / 256 != b / 256)) failures++;
        }
        for (size_t t = 0; t < n; t++) failures += seen[t] != 1;
    }
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
