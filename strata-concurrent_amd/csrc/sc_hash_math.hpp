// sc_hash_math.hpp - the parts of the hash kernels (sc_hash.hip) that hold on a host as on the device: constexpr
// functions and tables, compiled into the kernels and, by the CPU tests, into a host program that compares them with the
// byte loop and plain searches.
#pragma once

#include <cstdint>

#include "sc_internal.hpp"

namespace sc {

constexpr uint64_t kFnvPrime = 1099511628211ull;
constexpr uint32_t kPrimeLow = 179u;   // kFnvPrime mod 256
// A lane's segment runs as two halves side by side.
constexpr int kPairBytes = 128, kHalfWords = kPairBytes / 4;

// ---- the sum on the matrix cores -------------------------------------------------------------------------------------
// A run of bytes adds sum over n of d_n p^(E_n) to the hash, d_n = x_n - l_n, x_n = l_n ^ b_n, E_n the bytes from n to
// the input's end.  The machine's product 179 x_n = lo_n + 256 hi_n holds both: lo_n is l_(n+1), and
// x_n = (lo_n + 256 hi_n) / 179, exact as a multiplication by the inverse of 179 modulo 2^64.  So
//     sum d_n p^(E_n) = sum lo_n u(E_n) + sum hi_n v(E_n) + (low byte after the run) p^(E_end) - (low byte before) p^(E_0),
//     u(E) = p^E / 179 - p^(E-1),   v(E) = 256 p^E / 179   (mod 2^64),
// linear in the bytes of the products a lane's two machines leave in one register per step.  With the weights as eight
// signed base-256 digits (balanced, so |digit| <= 128; the carry out of the top digit is a multiple of 2^64 and drops)
// it is a product of 8-bit matrices: v_mfma_i32_16x16x64_i8, four steps' products per lane as A, the digits as B.  The
// products' bytes are offset by -128 (one xor) to be signed, which adds a constant.  Row i of the result sums lanes
// i, i + 16, i + 32, i + 48, whose distance is in the weights, and column j digit j; columns 0-7 hold the weights of an
// even word and columns 8-15 those of the odd word after it, so one B serves two multiplications.  Every sum is below
// 1024 * 2^14 in magnitude, so exact in 32 bits.
// Against two packed 16-bit dot products per byte pair and digit (v_dot2_i32_i16, four 16-bit digits, 9 operations per
// two bytes) this leaves the vector units four operations per two bytes.
constexpr uint64_t prime_pow_of(uint64_t e) {
    uint64_t r = 1, b = kFnvPrime;
    for (; e; e >>= 1, b *= b)
        if (e & 1) r *= b;
    return r;
}
constexpr uint64_t inverse_of(uint64_t a) {   // modulo 2^64, a odd: Newton's iteration doubles the correct bits
    uint64_t x = a;
    for (int i = 0; i < 6; ++i) x *= 2u - a * x;
    return x;
}
constexpr uint64_t kInv179 = inverse_of(kPrimeLow);
static_assert(kInv179 * kPrimeLow == 1u, "the inverse of 179 modulo 2^64");
constexpr uint64_t kPrimeInv = inverse_of(kFnvPrime);
// u(E) and v(E) from p^E.
constexpr uint64_t weight_lo(uint64_t pe) { return kInv179 * pe - kPrimeInv * pe; }
constexpr uint64_t weight_hi(uint64_t pe) { return 256u * kInv179 * pe; }
struct SumWeights {
    uint32_t w[kHalfWords / 2][64][4];   // [word pair][lane][step]: the lane's B operand, bytes (A lo, A hi, B lo, B hi)
};
constexpr SumWeights sum_weights() {
    SumWeights t{};
    // p^(E + 4096 (3 - q)) of byte c of half A, for lane group q; half B's is 128 bytes nearer the end
    for (int q = 0; q < 4; ++q) {
        uint64_t pa = prime_pow_of(uint64_t(2 * kPairBytes) + 4096u * uint64_t(3 - q));
        uint64_t pb = prime_pow_of(uint64_t(kPairBytes) + 4096u * uint64_t(3 - q));
        for (int c = 0; c < kPairBytes; ++c) {
            uint64_t v[4] = {weight_lo(pa), weight_hi(pa), weight_lo(pb), weight_hi(pb)};
            const int word = c / 4, column = (word & 1) * 8;
            for (int digit = 0; digit < 8; ++digit) {
                uint32_t bytes = 0;
                for (int k = 0; k < 4; ++k) {
                    const uint64_t low = v[k] & 0xFFu;
                    bytes |= uint32_t(low) << (8 * k);
                    v[k] = (v[k] >> 8) + (low >= 128u ? 1u : 0u);   // the balanced digit's carry
                }
                t.w[word / 2][16 * q + column + digit][c % 4] = bytes;
            }
            pa *= kPrimeInv;
            pb *= kPrimeInv;
        }
    }
    return t;
}
// 128 times the sum of a segment's weights relative to its end: what offsetting its products' bytes takes away.
constexpr uint64_t offset_sum() {
    uint64_t sum = 0, pe = prime_pow_of(2 * kPairBytes);
    for (int c = 0; c < 2 * kPairBytes; ++c, pe *= kPrimeInv) sum += weight_lo(pe) + weight_hi(pe);
    return 128u * sum;
}
constexpr uint64_t kOffsetSum = offset_sum();
// Per lane l: p^(256 (63 - l)), which takes a segment's value from its end to the end of the wave's last segment, and
// 2^(8 (l mod 8)) p^(256 (12 - 4 (l / 16))), which does so for the lane's column and rows of the product.
struct LanePow {
    uint64_t v[64], col[64];
};
constexpr LanePow lane_pow() {
    LanePow t{};
    for (int l = 0; l < 64; ++l) {
        t.v[l] = prime_pow_of(uint64_t(kFnvLaneBytes) * uint64_t(63 - l));
        t.col[l] = prime_pow_of(uint64_t(kFnvLaneBytes) * uint64_t(12 - 4 * (l / 16))) << (8 * (l % 8));
    }
    return t;
}

// s p^e modulo 2^64 for a signed 32-bit s: p^e as 2^32 hi + a signed low word.
template <uint64_t kPow>
__attribute__((always_inline)) constexpr uint64_t times_pow(int32_t s) {
    constexpr int32_t lo = int32_t(uint32_t(kPow));
    constexpr uint32_t hi = uint32_t(kPow >> 32) + (lo < 0 ? 1u : 0u);
    return uint64_t(int64_t(s) * int64_t(lo)) + (uint64_t(uint32_t(s) * hi) << 32);
}

// ---- maps of a level ----
// A level resolves kBits bits of the state, j .. j + kBits - 1.  A run's map of the level holds, for each of those bits and
// each start value of the level's lower ones, the term the run xors onto the bit: bit 0 the term of bit j, bits 1-2 those
// of bit j + 1 for start bit j = 0, 1, bits 3-6 those of bit j + 2, bits 7-14 those of bit j + 3.  The terms of bit i start
// at 2^i - 1 and are indexed by the start bits before it as one number, the lowest bit of the state first (most
// significant).  0 is the identity.
template <int kBits>
constexpr uint32_t map_mask() { return (1u << ((1u << kBits) - 1u)) - 1u; }
template <int kBits>
constexpr uint32_t state_mask() { return (1u << kBits) - 1u; }

// A run's map from its machines' end states: e[m] ended the machine started from the true lower bits, m in the level's
// lowest kBits - 2 bits and zeros above.  The top bit's terms for a set start bit below it follow from that bit's own term,
// the parity of that bit over the run's bytes (`par`, the xor of the bytes) and the run's length (`odd`).
template <int kJ, int kBits>
__attribute__((always_inline)) constexpr uint32_t map_of(const uint32_t (&e)[1 << (kBits - 2)], uint32_t par, uint32_t odd) {
    const uint32_t flip = ((par >> (kJ + kBits - 2)) & 1u) ^ odd;
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < kBits; ++i)
#pragma unroll
        for (int at = 0; at < (1 << i); ++at) {   // the start bits before bit i, the first most significant
            int machine = 0;
#pragma unroll
            for (int k = 0; k < i && k < kBits - 2; ++k) machine |= ((at >> (i - 1 - k)) & 1) << k;
            uint32_t term = (e[machine] >> (kJ + i)) & 1u;
            if (i == kBits - 1 && (at & 1)) term ^= ((e[machine] >> (kJ + kBits - 2)) & 1u) ^ flip;
            m |= term << ((1 << i) - 1 + at);
        }
    return m;
}

// The state after a map.
template <int kBits>
__attribute__((always_inline)) constexpr uint32_t apply(uint32_t m, uint32_t st) {
    uint32_t out = st, at = 0;
#pragma unroll
    for (int i = 0; i < kBits; ++i) {
        out ^= ((m >> ((1u << i) - 1u + at)) & 1u) << i;
        at = 2u * at + ((st >> i) & 1u);
    }
    return out;
}

// g after f.  `at` are the start bits before bit kBit in f, `gat` what they have become where g starts; the top bit's
// terms are taken two at a time, g's pair swapped where f flips the bit below.
template <int kBits, int kBit = 0>
__attribute__((always_inline)) constexpr uint32_t compose(uint32_t g, uint32_t f, uint32_t at = 0, uint32_t gat = 0) {
    constexpr uint32_t base = (1u << kBit) - 1u, next = (2u << kBit) - 1u;
    const uint32_t t = (f >> (base + at)) & 1u;
    uint32_t r = (t ^ ((g >> (base + gat)) & 1u)) << (base + at);
    if constexpr (kBit + 2 == kBits) {
        const uint32_t pair = (g >> (next + 2u * gat)) & 3u, swapped = (pair >> 1) | ((pair & 1u) << 1);
        r |= (((f >> (next + 2u * at)) & 3u) ^ (t ? swapped : pair)) << (next + 2u * at);
    } else {
        r |= compose<kBits, kBit + 1>(g, f, 2u * at, 2u * gat + t) |
             compose<kBits, kBit + 1>(g, f, 2u * at + 1u, 2u * gat + (t ^ 1u));
    }
    return r;
}

// ---- powers of the prime ----
// p^(2^k), p^(-2^k) and p^k.
struct FinishPow {
    uint64_t square[64], back[16], small[256];
};
constexpr FinishPow finish_pow() {
    FinishPow t{};
    uint64_t a = kFnvPrime, b = kPrimeInv, c = 1;
    for (int k = 0; k < 64; ++k, a *= a) t.square[k] = a;
    for (int k = 0; k < 16; ++k, b *= b) t.back[k] = b;
    for (int k = 0; k < 256; ++k, c *= kFnvPrime) t.small[k] = c;
    return t;
}

// (p^65536)^k as a product of one entry per byte of k: what a workgroup's sum is worth k whole 64 KiB before the last.
struct GroupPow {
    uint64_t v[4][256];
};
constexpr GroupPow group_pows() {
    GroupPow t{};
    uint64_t step = prime_pow_of(uint64_t(kFnvGroupBytes));
    for (int i = 0; i < 4; ++i) {
        uint64_t x = 1;
        for (int k = 0; k < 256; ++k, x *= step) t.v[i][k] = x;
        step = x;
    }
    return t;
}

// ---- the extents of a gathered payload ----
// The extents [first, first + size) that hold a payload byte, narrowed 64 at a time: lane l samples the end of the last
// extent of its share of the span, and the share after those that end at or before the byte is the next span.  A table of
// n extents takes ceil(log64 n) dependent reads.  (A share walked 64 ends at a time instead took n / 4096: 805 MB in 196 605
// extents gathered and hashed in 691 us, now in 546; up to 4096 extents, two reads at most, both take the same.)
struct ExtentSpan {
    uint32_t first, size;
    constexpr uint32_t share() const { return size / 64u + (size % 64u ? 1u : 0u); }
    // the extent lane `lane` samples (no sum here passes the last extent's index, so none wraps)
    constexpr uint32_t sample(uint32_t lane) const {
        const uint32_t each = share(), at = lane * each < size ? lane * each : size - 1u;
        return first + at + (each - 1u < size - 1u - at ? each - 1u : size - 1u - at);
    }
    // `passed` lanes sampled an end at or before the byte (never all: the last extent's end lies past it)
    constexpr void narrow(uint32_t passed) {
        const uint32_t each = share(), skip = passed * each < size ? passed * each : size - 1u;
        first += skip;
        size = each < size - skip ? each : size - skip;
    }
};

}  // namespace sc
