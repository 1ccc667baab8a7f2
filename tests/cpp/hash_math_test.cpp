// The hash kernels' host-evaluable parts (csrc/sc_hash_math.hpp, the header the kernels are compiled from) against plain
// loops.  `hash_math_test <name>` runs one test; it prints the first difference and returns 1, or returns 0.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "sc_hash_math.hpp"

namespace {

#define REQUIRE(cond, ...)                                   \
    do {                                                     \
        if (!(cond)) {                                       \
            std::printf("%s:%d: %s: ", __FILE__, __LINE__, #cond); \
            std::printf(__VA_ARGS__);                        \
            std::printf("\n");                               \
            return 1;                                        \
        }                                                    \
    } while (0)

// The search of a workgroup's first extent: 64 lanes sampling `end_of(i)`, the end of extent i.
template <typename End>
int find(uint32_t n, uint64_t byte, const End& end_of, uint32_t want) {
    sc::ExtentSpan span{0u, n};
    uint32_t looks = 0, most = 1;
    for (uint64_t reach = 64; reach < n; reach *= 64) ++most;
    do {
        uint32_t passed = 0;
        for (uint32_t lane = 0; lane < 64; ++lane) {
            const uint32_t at = span.sample(lane);
            REQUIRE(at < n, "lane %u of a table of %u samples %u", lane, n, at);
            if (end_of(at) <= byte) ++passed;
        }
        span.narrow(passed);
        ++looks;
        REQUIRE(looks <= most, "a table of %u took more than %u looks", n, most);
    } while (span.size > 1u);
    REQUIRE(span.first == want, "byte %llu of %u extents: %u, not %u", (unsigned long long) byte, n, span.first, want);
    return 0;
}

int extents() {
    std::mt19937_64 rng(1);
    // tables of one size of extent, up to the most a map holds
    for (uint64_t n : {1ull, 2ull, 63ull, 64ull, 65ull, 127ull, 128ull, 129ull, 4095ull, 4096ull, 4097ull, 65535ull, 196605ull,
                       262144ull, 262145ull, (1ull << 31) - 1, 1ull << 31, (1ull << 32) - 64, (1ull << 32) - 63,
                       (1ull << 32) - 1}) {
        const auto end_of = [](uint64_t i) { return (i + 1) * 48; };
        for (int k = 0; k < 60; ++k) {
            const uint64_t e = k == 0 ? 0 : k == 1 ? n - 1 : k < 20 ? std::min<uint64_t>(n - 1, uint64_t(k) * 63) : rng() % n;
            for (uint64_t byte : {e * 48, e * 48 + 47})
                if (find(uint32_t(n), byte, end_of, uint32_t(e))) return 1;
        }
    }
    // ragged ones
    for (int t = 0; t < 200; ++t) {
        const uint32_t n = uint32_t(1 + rng() % (t % 4 ? 300 : 20000));
        std::vector<uint64_t> ends;
        uint64_t at = 0;
        for (uint32_t i = 0; i < n; ++i) ends.push_back(at += 16 * (1 + rng() % (rng() % 8 ? 40 : 9000)));
        for (int k = 0; k < 40; ++k) {
            const uint64_t byte = rng() % at;
            uint32_t want = 0;
            while (ends[want] <= byte) ++want;
            if (find(n, byte, [&](uint32_t i) { return ends[i]; }, want)) return 1;
        }
    }
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    const struct { const char* name; int (*run)(); } tests[] = {{"extents", extents}};
    for (const auto& t : tests)
        if (argc == 2 && !std::strcmp(argv[1], t.name)) return t.run();
    std::printf("usage: hash_math_test <test>\n");
    return 2;
}
