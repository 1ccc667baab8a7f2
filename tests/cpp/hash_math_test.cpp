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

// The byte loop, its low byte alone, and p^e by its definition.
uint64_t fnv(uint64_t h, const std::vector<uint8_t>& data, size_t from = 0, size_t to = SIZE_MAX) {
    for (size_t i = from; i < std::min(to, data.size()); ++i) h = (h ^ data[i]) * 1099511628211ull;
    return h;
}
uint32_t low_byte(uint32_t l, const uint8_t* p, size_t n) {
    for (size_t i = 0; i < n; ++i) l = ((l ^ p[i]) * 179u) & 0xFFu;
    return l;
}
std::vector<uint8_t> bytes_of(std::mt19937_64& rng, size_t n, int kind) {
    std::vector<uint8_t> v(n);
    const uint8_t mask = kind == 1 ? uint8_t(rng()) : 0xFF;   // some bits constant
    for (uint8_t& b : v) b = kind == 2 ? 0xFF : kind == 3 ? 0 : uint8_t(rng()) & mask;
    return v;
}

// ---- the levels: a run's map takes every start of the level to its end, and maps compose in the order of their runs
template <int kJ, int kBits>
uint32_t run_map(uint32_t low, const uint8_t* p, size_t n) {
    uint32_t e[1 << (kBits - 2)], par = 0;
    for (uint32_t m = 0; m < (1u << (kBits - 2)); ++m) e[m] = low_byte(low | (m << kJ), p, n);
    for (size_t i = 0; i < n; ++i) par ^= p[i];
    return sc::map_of<kJ, kBits>(e, par, uint32_t(n & 1));
}
template <int kJ, int kBits>
int level() {
    std::mt19937_64 rng(kJ * 8 + kBits);
    for (int t = 0; t < 2000; ++t) {
        const std::vector<uint8_t> v = bytes_of(rng, rng() % 200, t % 4);
        const uint32_t low = uint32_t(rng()) & ((1u << kJ) - 1u);
        const size_t cut = rng() % (v.size() + 1);
        const uint32_t whole = run_map<kJ, kBits>(low, v.data(), v.size());
        const uint32_t a = run_map<kJ, kBits>(low, v.data(), cut);
        const uint32_t b = run_map<kJ, kBits>(low_byte(low, v.data(), cut) & ((1u << kJ) - 1u), v.data() + cut, v.size() - cut);
        REQUIRE(whole <= sc::map_mask<kBits>(), "level %d of %d bits: map %x", kJ, kBits, whole);
        REQUIRE(sc::compose<kBits>(b, a) == whole, "level %d of %d bits, %zu bytes cut at %zu", kJ, kBits, v.size(), cut);
        REQUIRE(sc::compose<kBits>(whole, 0u) == whole && sc::compose<kBits>(0u, whole) == whole, "0 is the identity");
        for (uint32_t st = 0; st <= sc::state_mask<kBits>(); ++st) {
            const uint32_t want = (low_byte(low | (st << kJ), v.data(), v.size()) >> kJ) & sc::state_mask<kBits>();
            REQUIRE(sc::apply<kBits>(whole, st) == want, "level %d of %d bits from %u", kJ, kBits, st);
        }
    }
    return 0;
}
int levels() { return level<0, 4>() || level<4, 4>() || level<0, 3>() || level<3, 3>() || level<6, 2>(); }

// ---- the sum of a wave's 64 segments: the products' bytes times the weights' digits, as the matrix instruction pairs
// them (row and column of a lane's operands lane % 16, results in rows 4 (lane / 16) + 0 .. 3 of column lane % 16)
int sums() {
    std::mt19937_64 rng(2);
    static const sc::SumWeights weights = sc::sum_weights();
    static const sc::LanePow pow = sc::lane_pow();
    for (int t = 0; t < 8; ++t) {
        const std::vector<uint8_t> v = bytes_of(rng, 64 * 256, t % 4);
        const uint64_t h0 = rng();
        std::vector<uint32_t> start(65), mid(64);
        start[0] = uint32_t(h0) & 0xFFu;
        static int64_t c[2][16][16];   // of even and of odd words
        std::memset(c, 0, sizeof c);
        for (int lane = 0; lane < 64; ++lane) {
            const uint8_t* p = v.data() + lane * 256;
            mid[size_t(lane)] = low_byte(start[size_t(lane)], p, 128);
            start[size_t(lane) + 1] = low_byte(mid[size_t(lane)], p + 128, 128);
            uint32_t a = start[size_t(lane)], b = mid[size_t(lane)];
            for (int k = 0; k < sc::kHalfWords; ++k)
                for (int i = 0; i < 4; ++i) {
                    const uint32_t pa = (a ^ p[4 * k + i]) * 179u, pb = (b ^ p[128 + 4 * k + i]) * 179u;
                    a = pa & 0xFFu, b = pb & 0xFFu;
                    const uint32_t m = (pa | (pb << 16)) ^ 0x80808080u;
                    for (int column = 0; column < 16; ++column) {
                        const uint32_t w = weights.w[k / 2][16 * (lane / 16) + column][i];
                        for (int s = 0; s < 32; s += 8)
                            c[k & 1][lane % 16][column] += int64_t(int8_t(m >> s)) * int8_t(w >> s);
                    }
                }
        }
        uint64_t sum = 0;
        constexpr uint64_t p1 = sc::prime_pow_of(256), p2 = p1 * p1, p3 = p2 * p1;
        for (int lane = 0; lane < 64; ++lane) {
            int32_t s[4];
            for (int r = 0; r < 4; ++r) {
                const int64_t x = c[(lane >> 3) & 1][4 * (lane / 16) + r][lane % 16];
                REQUIRE(x >= -(1 << 24) && x <= (1 << 24), "a sum of %lld", (long long) x);
                s[r] = int32_t(x);
            }
            const uint64_t rows = sc::times_pow<p3>(s[0]) + sc::times_pow<p2>(s[1]) + sc::times_pow<p1>(s[2]) + uint64_t(int64_t(s[3]));
            const uint64_t ends = uint64_t(start[size_t(lane) + 1]) - sc::times_pow<p1>(int32_t(start[size_t(lane)])) + sc::kOffsetSum;
            sum += rows * pow.col[lane] + ends * pow.v[lane];
        }
        REQUIRE(h0 * sc::prime_pow_of(16384) + sum == fnv(h0, v), "the wave's sum, data %d", t);
    }
    for (int t = 0; t < 10000; ++t) {
        const int32_t s = t < 4 ? int32_t(t - 2) : t == 4 ? INT32_MIN : t == 5 ? INT32_MAX : int32_t(rng());
        constexpr uint64_t a = sc::prime_pow_of(256), b = sc::prime_pow_of(1);
        REQUIRE(sc::times_pow<a>(s) == uint64_t(int64_t(s)) * a && sc::times_pow<b>(s) == uint64_t(int64_t(s)) * b, "%d", s);
    }
    return 0;
}

// ---- the powers that bring the sums together
int powers() {
    std::mt19937_64 rng(3);
    static const sc::GroupPow group = sc::group_pows();
    static const sc::FinishPow finish = sc::finish_pow();
    for (int t = 0; t < 20000; ++t) {
        const uint32_t k = t < 600 ? uint32_t(t) : t < 632 ? 1u << (t - 600) : uint32_t(rng() >> (32 + rng() % 32));
        uint64_t got = 1;
        for (int i = 0; i < 4; ++i) got *= group.v[i][(k >> (8 * i)) & 255u];
        REQUIRE(got == sc::prime_pow_of(uint64_t(sc::kFnvGroupBytes) * k), "%u pieces", k);
        const uint64_t n = rng() >> (rng() % 64);
        uint64_t up = 1, back = 1;
        for (int b = 0; b < 64; ++b) up *= (n >> b) & 1u ? finish.square[b] : 1u;
        for (int b = 0; b < 16; ++b) back *= (n >> b) & 1u ? finish.back[b] : 1u;
        REQUIRE(up == sc::prime_pow_of(n), "p^%llu", (unsigned long long) n);
        REQUIRE(back * sc::prime_pow_of(n & 0xFFFFu) == 1u, "p^-%llu", (unsigned long long) (n & 0xFFFFu));
    }
    for (uint64_t k = 0; k < 256; ++k) REQUIRE(finish.small[k] == sc::prime_pow_of(k), "p^%llu", (unsigned long long) k);
    // whole pieces' sums, each relative to the end of its 64 KiB, and the last partial one's, closed into the hash
    for (size_t n : {size_t(256), size_t(65536 - 256), size_t(65536), size_t(65536 + 256), size_t(3 * 65536 + 512)}) {
        const std::vector<uint8_t> v = bytes_of(rng, n, 0);
        const uint64_t h0 = rng();
        const uint32_t pieces = uint32_t((n + 65535) / 65536);
        uint64_t whole = 0, h = h0;
        for (uint32_t g = 0; g < pieces; ++g) {
            const size_t from = size_t(g) * 65536, to = std::min(from + 65536, n);
            const uint64_t end = fnv(h, v, from, to), sum = end - h * sc::prime_pow_of(to - from);   // relative to `to`
            const uint32_t rest = pieces - 1 - g;
            uint64_t worth = 1;
            for (int i = 0; i < 4; ++i) worth *= group.v[i][(rest >> (8 * i)) & 255u];
            whole += sum * sc::prime_pow_of(from + 65536 - to) * worth;
            h = end;
        }
        const uint32_t past = uint32_t((65536 - n % 65536) % 65536);
        uint64_t back = 1;
        for (int b = 0; b < 16; ++b) back *= (past >> b) & 1u ? finish.back[b] : 1u;
        REQUIRE(h0 * sc::prime_pow_of(n) + whole * back == fnv(h0, v), "%zu bytes", n);
    }
    return 0;
}

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
    const struct { const char* name; int (*run)(); } tests[] = {{"levels", levels}, {"sums", sums}, {"powers", powers},
                                                                {"extents", extents}};
    for (const auto& t : tests)
        if (argc == 2 && !std::strcmp(argv[1], t.name)) return t.run();
    std::printf("usage: hash_math_test <test>\n");
    return 2;
}
