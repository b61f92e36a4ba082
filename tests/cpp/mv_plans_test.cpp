// Minimum variance planned for different shares of the LDS (as a batch plans
// its queues), with and without room for the pre-delay's tables, gives one
// image, bit for bit.  Prints one line per configuration; exits with the number of failures.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <set>
#include <vector>

#include "mv_launch.hpp"
#include "supra_bf.h"

using namespace supra_amd;

namespace {

uint32_t state = 1;
float uniform() {
    state = state * 1664525u + 1013904223u;
    return static_cast<float>(state >> 8) * 0x1p-24f;
}

// [scanline][channel][depth]; apertures of every length, so that windows of few
// and of many sub-array vectors alternate, and two empty depths.
std::vector<float> signals(uint32_t n_rx, uint32_t n_ch, uint32_t n_d, uint32_t L) {
    std::vector<float> x(static_cast<size_t>(n_rx) * n_ch * n_d, 0.0f);
    for (uint32_t s = 0; s < n_rx; s++)
        for (uint32_t d = 0; d < n_d; d++) {
            const bool few = (d / 21) % 2 != 0;
            const uint32_t len = few ? std::min(n_ch, L) : 1 + static_cast<uint32_t>(uniform() * static_cast<float>(n_ch));
            const uint32_t first = static_cast<uint32_t>(uniform() * static_cast<float>(n_ch - std::min(len, n_ch) + 1));
            for (uint32_t c = first; c < std::min(n_ch, first + len); c++)
                x[(static_cast<size_t>(s) * n_ch + c) * n_d + d] = d % 37 == 36 ? 0.0f : 200.0f * (uniform() - 0.5f);
        }
    return x;
}

#define CHECK(call)                                                                             \
    do {                                                                                        \
        const hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess) {                                                                 \
            std::printf("%s: %s\n", #call, hipGetErrorString(e_));                              \
            return 100;                                                                         \
        }                                                                                       \
    } while (0)

int run(uint32_t n_ch, uint32_t n_d, uint32_t L, uint32_t T, bool means) {
    const uint32_t n_rx = 3;
    const std::vector<float> x = signals(n_rx, n_ch, n_d, L);
    const size_t out_bytes = static_cast<size_t>(n_rx) * n_d * sizeof(float);
    float *dx = nullptr, *dout = nullptr;
    CHECK(hipMalloc(&dx, x.size() * sizeof(float)));
    CHECK(hipMalloc(&dout, out_bytes));
    CHECK(hipMemcpy(dx, x.data(), x.size() * sizeof(float), hipMemcpyHostToDevice));
    std::vector<float> first(n_rx * n_d), img(n_rx * n_d);
    std::set<uint32_t> tiles;
    int failures = 0, plans = 0;
    for (int plan = 0; plan < 16; plan++) {
        const uint32_t share = 1 + plan % 8;
        MvArgs a;
        std::memset(&a, 0, sizeof(a));
        a.x = dx;
        a.out = dout;
        if (plan >= 8) a.g.rf = dx;     // (planned, not launched, as a fused call)
        size_t lds = 0;
        if (mv_prepare(a, n_rx, n_ch, n_d, L, T, 1.5, means ? 1 : 0, 0.1, false, 163840u / share - 64u, &lds) != SUPRA_OK ||
            !a.block)
            continue;      // does not fit
        plans++;
        CHECK(hipMemset(dout, 0xff, out_bytes));
        CHECK(launch_mv_block(a, SUPRA_FLOAT32, false, lds, nullptr));
        CHECK(hipMemcpy(img.data(), dout, out_bytes, hipMemcpyDeviceToHost));
        tiles.insert(a.tile);
        if (plan == 0) first = img;
        failures += std::memcmp(first.data(), img.data(), out_bytes) != 0;
    }
    CHECK(hipFree(dx));
    CHECK(hipFree(dout));
    failures += plans < 2;
    std::printf("L=%u T=%u channels=%u depths=%u means=%d: tiles", L, T, n_ch, n_d, means);
    for (uint32_t t : tiles) std::printf(" %u", t);
    std::printf(", %d plans, %d failures\n", plans, failures);
    std::fflush(stdout);
    return failures;
}

}  // namespace

int main() {
    int failures = 0;
    failures += run(128, 90, 64, 5, false);
    failures += run(128, 90, 64, 2, false);
    failures += run(96, 61, 48, 3, true);
    failures += run(256, 70, 32, 5, false);
    failures += run(256, 70, 32, 9, true);
    failures += run(200, 7, 64, 4, false);
    failures += run(256, 75, 16, 12, true);
    failures += run(128, 40, 8, 0, false);
    failures += run(48, 4200, 16, 4, false);     // tall tiles
    failures += run(40, 6200, 8, 18, true);
    failures += run(170, 8200, 5, 10, false);
    return failures;
}
