// Host check of the division by three of the mean flow (mr-lbm_amd/csrc/linear.h):
// the quotient of every 32-bit value tried is that of the division, infinities
// and NaN among them. Prints "ok" and exits 0 on success.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "../mr-lbm_amd/csrc/linear.h"

int main() {
    int failures = 0;
    auto check = [&](uint32_t bits) {
        float f;
        std::memcpy(&f, &bits, 4);
        const double got = mrlbm::third((double)f), want = (double)f / 3.0;
        failures += std::isnan(want) ? !std::isnan(got) : got != want;
    };
    for (uint32_t e = 0; e < 512; e++)  // every sign and exponent
        for (uint32_t m : {0u, 1u, 2u, 3u, 0x2AAAAAu, 0x400000u, 0x555555u, 0x7FFFFEu, 0x7FFFFFu}) check(e << 23 | m);
    uint32_t x = 1;
    for (int k = 0; k < 4000000; k++) check(x = x * 1664525u + 1013904223u);
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
