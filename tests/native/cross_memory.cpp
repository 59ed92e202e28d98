// A crossover plan whose segment partials would not fit the device memory takes
// fewer segments, and is refused only when one segment's do not fit either
// (fake_hip.cpp: no device).  2,560 x 256 pairs x 9,000 bars, by the plan's own
// count of 28 bytes per pair and segment, 40 per pair and 8 per row and bar:
// 358 MB in eight segments, 229 in one.
#include <cstdio>
#include <vector>

#include "fake_hip.h"
#include "vta.h"

namespace {
vta_alma_batch_range range(size_t p0, size_t p1, double o1) {
    vta_alma_batch_range r{};
    r.period = {p0, p1, 1};
    r.offset = {0.0, o1, 0.1};
    r.sigma = {6.0, 6.0, 0.0};
    return r;
}
}  // namespace

int main() {
    vta_ctx *ctx = nullptr;
    if (vta_ctx_create(0, &ctx) != VTA_OK) return 2;
    std::vector<float> x(9000);
    for (size_t i = 0; i < x.size(); ++i) x[i] = 100.0f + (float)(i % 97);
    const vta_alma_batch_range fast = range(5, 260, 0.9), slow = range(5, 260, 0.0);
    const size_t mb = 1000000, headroom = 64u << 20;
    for (const size_t free_mb : {2000, 450, 300, 100}) {
        fake_hip_memory(free_mb * mb + headroom);
        vta_double_alma_plan *plan = nullptr;
        const vta_status st = vta_double_alma_plan_create(ctx, x.data(), x.size(), &fast, &slow, &plan);
        std::printf("%zu MB: %d %s\n", free_mb, (int)st, vta_last_error());
        if ((st == VTA_OK) != (free_mb > 200)) return 1;
        if (st == VTA_OK && vta_last_error()[0]) return 1;   // (nothing left of the first tries)
        if (plan) vta_double_alma_plan_destroy(plan);
    }
    vta_ctx_destroy(ctx);
    std::puts("ok");
    return 0;
}
