// Admission of the request server under a full memory budget, without a device
// (fake_hip.cpp).  One scenario per run, named by argv[1]; exit status 0 when
// it holds.  Built with AddressSanitizer by tests/test_host_memory.py.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "fake_hip.h"
#include "vta.h"

namespace {

constexpr size_t kBars = 100000, kRow = kBars * sizeof(float);   // 400,000 bytes

#define CHECK(c)                                                        \
    do {                                                                \
        if (!(c)) {                                                     \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);         \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

struct Server {
    vta_server *s = nullptr;
    std::vector<float> x = std::vector<float>(kBars, 1.0f);
    Server(size_t rows) {
        // (a few bytes of room beside whole rows)
        CHECK(vta_server_create(0, 1, rows * kRow + 1024, &s) == VTA_OK);
    }
    ~Server() { vta_server_destroy(s); }
    // An EMA (or, hlc, ADX) request of `rows` output rows on series `key`.
    uint64_t submit(uint64_t key, size_t rows, bool hlc = false) {
        vta_request r{};
        r.kind = hlc ? VTA_REQ_ADX : VTA_REQ_EMA;
        r.cache = 1;
        r.series_key = key;
        r.close = x.data();
        if (hlc) r.high = r.low = x.data();
        r.len = kBars;
        r.period.start = 2;
        r.period.end = 2 + rows - 1;
        r.period.step = 1;
        uint64_t id = 0;
        CHECK(vta_server_submit(s, &r, &id) == VTA_OK);
        return id;
    }
    int wait(uint64_t id) {
        vta_result res{};
        const vta_status v = vta_server_wait(s, id, 20000, &res);
        return v == VTA_OK ? res.status : v;
    }
    int serve(uint64_t key, size_t rows, bool hlc = false) {
        const uint64_t id = submit(key, rows, hlc);
        const int st = wait(id);
        CHECK(vta_server_release(s, id) == VTA_OK);
        return st;
    }
    vta_server_stats stats() {
        vta_server_stats st{};
        CHECK(vta_server_get_stats(s, &st) == VTA_OK);
        CHECK(st.peak_in_use <= st.budget);
        return st;
    }
};

// A hit whose own series is the least recently used of two: the other one is
// evicted for its outputs.
void hit_evicts_another() {
    Server v(4);
    CHECK(v.serve(1, 1) == VTA_OK);
    CHECK(v.serve(2, 1) == VTA_OK);
    CHECK(v.stats().cached_series == 2);
    const uint64_t id = v.submit(1, 3);
    CHECK(v.wait(id) == VTA_OK);
    CHECK(v.stats().cached_series == 1);
    CHECK(v.stats().in_use == 4 * kRow);
    CHECK(vta_server_release(v.s, id) == VTA_OK);
    CHECK(v.stats().in_use == kRow);
    CHECK(v.serve(1, 3) == VTA_OK);          // still the same, uploaded series
    CHECK(v.stats().cached_series == 1);
}

// A hit whose own series is the only one to evict, and whose outputs do not
// fit beside it: it can never be served.
void hit_never_fits() {
    Server v(3);
    CHECK(v.serve(1, 1) == VTA_OK);
    CHECK(v.serve(1, 3) == VTA_ERR_OUT_OF_MEMORY);
    CHECK(v.serve(1, 2) == VTA_OK);          // the next request is not held up
    CHECK(v.stats().in_use <= kRow);
}

// A hit on a series cached with high and low, which its outputs do not fit
// beside, though they fit beside the close alone: served as a miss.
void hit_served_as_miss() {
    Server v(5);
    CHECK(v.serve(1, 1, true) == VTA_OK);
    CHECK(v.stats().in_use == 3 * kRow);
    const uint64_t id = v.submit(1, 4);
    CHECK(v.wait(id) == VTA_OK);
    CHECK(v.stats().in_use == 5 * kRow);
    CHECK(v.stats().cached_series == 1);
    CHECK(vta_server_release(v.s, id) == VTA_OK);
    CHECK(v.stats().in_use == kRow);
}

// A hit that fits only once an earlier result is released waits for it, and
// its series stays evictable afterwards.
void hit_waits_for_release() {
    Server v(4);
    const uint64_t held = v.submit(1, 2);
    CHECK(v.wait(held) == VTA_OK);
    const uint64_t id = v.submit(1, 2);
    vta_result res{};
    CHECK(vta_server_wait(v.s, id, 200, &res) == VTA_ERR_TIMEOUT);
    CHECK(v.stats().queued == 1);
    CHECK(vta_server_release(v.s, held) == VTA_OK);
    CHECK(v.wait(id) == VTA_OK);
    CHECK(vta_server_release(v.s, id) == VTA_OK);
    CHECK(v.serve(2, 3) == VTA_OK);          // evicts series 1
    CHECK(v.stats().cached_series == 1);
    CHECK(v.stats().in_use == kRow);
}

// The same while a slot collects a pack: hits of series that only eviction of
// each other's would make room for.
void pack_of_hits() {
    Server v(8);
    for (uint64_t k = 1; k <= 4; ++k) CHECK(v.serve(k, 1) == VTA_OK);
    CHECK(v.stats().in_use == 4 * kRow);
    fake_hip_gate(true);
    const uint64_t first = v.submit(9, 2);   // evicts none or some, then waits
    fake_hip_wait_for_waiter();
    std::vector<uint64_t> ids;
    for (uint64_t k = 1; k <= 4; ++k) ids.push_back(v.submit(k, 2));
    fake_hip_gate(false);
    CHECK(v.wait(first) == VTA_OK);
    CHECK(vta_server_release(v.s, first) == VTA_OK);
    for (const uint64_t id : ids) {
        CHECK(v.wait(id) == VTA_OK);
        CHECK(vta_server_release(v.s, id) == VTA_OK);
    }
    CHECK(v.stats().queued == 0);
}

// Free memory in pieces between results that the client holds: a request that
// the budget holds, but no piece, waits for its neighbours' release.
void fragmented_arena() {
    constexpr size_t kSmall = 5, kN = 128;               // 2 MB results
    constexpr size_t kLarge = 300;                       // (the arena's end holds 208 rows)
    Server v(kN * kSmall + 1);
    std::vector<uint64_t> ids;
    for (size_t i = 0; i < kN; ++i) ids.push_back(v.submit(1, kSmall));
    for (const uint64_t id : ids) CHECK(v.wait(id) == VTA_OK);
    for (size_t i = 0; i < kN; i += 2) CHECK(vta_server_release(v.s, ids[i]) == VTA_OK);
    CHECK(v.stats().in_use + kLarge * kRow <= v.stats().budget);
    const uint64_t id = v.submit(1, kLarge);
    vta_result res{};
    CHECK(vta_server_wait(v.s, id, 300, &res) == VTA_ERR_TIMEOUT);
    CHECK(v.stats().queued == 1);
    for (size_t i = 1; i < kN; i += 2) CHECK(vta_server_release(v.s, ids[i]) == VTA_OK);
    CHECK(v.wait(id) == VTA_OK);
    CHECK(vta_server_release(v.s, id) == VTA_OK);
    CHECK(v.stats().in_use <= kRow);
}

const struct {
    const char *name;
    void (*run)();
} kScenarios[] = {{"hit_evicts_another", hit_evicts_another},
                  {"hit_never_fits", hit_never_fits},
                  {"hit_served_as_miss", hit_served_as_miss},
                  {"hit_waits_for_release", hit_waits_for_release},
                  {"pack_of_hits", pack_of_hits},
                  {"fragmented_arena", fragmented_arena}};

}  // namespace

int main(int argc, char **argv) {
    for (const auto &s : kScenarios)
        if (argc > 1 && std::strcmp(argv[1], s.name) == 0) {
            s.run();
            std::puts("ok");
            return 0;
        }
    return 2;
}
