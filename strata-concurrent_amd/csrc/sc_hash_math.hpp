// sc_hash_math.hpp - the parts of the hash kernels (sc_hash.hip) that hold on a host as on the device: constexpr
// functions, compiled into the kernels and, by the CPU tests, into a host program that compares them with plain loops.
#pragma once

#include <cstdint>

namespace sc {

// The extents [first, first + size) that hold a payload byte, narrowed 64 at a time: lane l samples the end of the last
// extent of its share of the span, and the share after those that end at or before the byte is the next span.  A table of
// n extents takes ceil(log64 n) dependent reads.  (A share walked 64 ends at a time instead took n / 4096: 805 MB in 196 605
// extents gathered and hashed in 691 us, now in 549; up to 4096 extents, two reads at most, both take the same.)
struct ExtentSpan {
    uint32_t first, size;
    constexpr uint32_t share() const { return size / 64u + (size % 64u ? 1u : 0u); }
    // the extent lane `lane` samples (64 bits: the last shares of a table near 2^32 extents end past 32)
    constexpr uint32_t sample(uint32_t lane) const {
        const uint64_t end = uint64_t(lane + 1u) * share();
        return first + (end < size ? uint32_t(end) : size) - 1u;
    }
    // `passed` lanes sampled an end at or before the byte (never all: the last extent's end lies past it)
    constexpr void narrow(uint32_t passed) {
        const uint32_t each = share(), skip = passed < 64u && passed * each < size ? passed * each : size - 1u;
        first += skip;
        size = each < size - skip ? each : size - skip;
    }
};

}  // namespace sc
