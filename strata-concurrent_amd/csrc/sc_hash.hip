// sc_hash.hip - FNV-1a 64 of a device buffer, bit-identical to the byte loop, computed in parallel.
//
// The engine's one content hash is FNV-1a 64: for every byte, h = (h ^ b) * p mod 2^64 with the prime
// p = 1099511628211 (the reference's fnv1a64, src/core/pinned.cu:594-601).  As written it is one long serial chain,
// about 1 GB/s on a CPU core, and the reference runs it twice over a multi-GB hand-off payload.  Two facts make the
// exact same value computable in parallel:
//
//   1. The low byte of the state is a finite-state machine of its own.  Multiplication mod 2^64 keeps the low 8 bits
//      a function of the low 8 bits, and xor with a byte touches only the low 8 bits, so
//          l' = ((l ^ b) * 179) mod 256          (179 = p mod 256).
//      Moreover bit j of l' depends only on bits 0..j of l and b (multiplication by an odd constant and xor are both
//      "triangular"), and it is bit j of l xor a term that involves only the lower bits:
//          l'_j = l_j ^ t_j,   t_j = b_j ^ bit_j(((l ^ b) mod 2^j) * 179).
//      So once bits 0..j-1 of the state are known at every position, bit j at every position is an exclusive xor
//      prefix of the t_j terms: a scan.  Eight levels of scans recover the low byte at every position.
//   2. With the low byte known, the rest is linear.  Writing h ^ b = h + d with d = (l ^ b) - l (a small signed
//      number), h_N = h_0 p^N + sum_n d_n p^(N-n) mod 2^64: independent per-segment Horner sums, folded with powers
//      of p in any order.
//
// The buffer is split into lane segments of kFnvLaneBytes bytes, a workgroup's 256 lanes covering 64 KiB, and the
// low byte is resolved in levels: bits 0-3 and 4-7, or, where no workgroup waits for another (a check given carries),
// bits 0-2, 3-5 and 6-7.  A level's map of a run of bytes takes the level's bits
// at the run's start to their values at its end, given the true lower bits.  The term of a bit depends only on the
// lower start bits, so the end value of a bit in a machine started from the true lower bits, with the bit itself 0,
// is the run's term for that bit.  The top two bits of a level need no machines of their own: flipping start bit i
// (the bits below it fixed) flips bit i at every position, which changes the term of bit i + 1 by the xor over the run
// of 1 ^ y_i, y_i being bit i of ((l ^ b) mod 2^i) * 179; and y_i = l_i ^ l'_i ^ b_i, so that xor is
//     (length mod 2) ^ (term of bit i) ^ (parity of bit i over the run's bytes).
// A level for bits j .. j + k - 1 therefore runs 2^(k-2) machines, one per value of the unknown start bits
// j .. j + k - 3.  Each lane runs its segment as two halves of 128 bytes side by side: both halves' machines share the
// multiplies (two 8-bit machines per 24-bit multiply, bytes 0 and 2; the lowest bits follow l' = (l ^ b) * 3 mod 16, so
// four machines share one register a byte each), each half's map comes from its machines and its byte parities, and the
// lane's map is the second half's after the first's.  Per level: the lanes ballot their maps, each workgroup forms
// its map of the k-bit state from them, finds its start state by a look-back over the workgroups before it, each
// lane derives its start bits from the workgroup's state and the ballots by counting the lanes before it, and its first
// half's map gives the bits at its midpoint.  After the last level every lane runs the full machine of both halves
// from their now complete start bytes, whose products the matrix cores sum with the powers of p; the workgroups' sums are
// added, and a last kernel adds h_0 p^N.  All of it is one kernel that reads the input once (the one-pass hash, below).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "sc_handoff.h"
#include "sc_hash_math.hpp"
#include "sc_internal.hpp"

namespace sc {
namespace {

using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using gu32x4 = __attribute__((address_space(1))) u32x4;

__device__ __forceinline__ uint64_t pow_prime(uint64_t e) {
    uint64_t r = 1, b = kFnvPrime;
    while (e) {
        if (e & 1) r *= b;
        b *= b;
        e >>= 1;
    }
    return r;
}

// The 16 dwords of one full, 16-byte aligned lane segment.
__device__ __forceinline__ void load_segment(const uint8_t* p, uint32_t (&w)[kFnvLaneBytes / 4]) {
#pragma unroll
    for (int k = 0; k < kFnvLaneBytes / 16; ++k) {
        const u32x4 v = *(const gu32x4*) (p + 16 * k);
        w[4 * k + 0] = v.x;
        w[4 * k + 1] = v.y;
        w[4 * k + 2] = v.z;
        w[4 * k + 3] = v.w;
    }
}

// Two low-byte machines side by side, in bytes 0 and 2 of `x`: xor the byte into both, drop the products' high
// bytes, one 24-bit multiply (byte 0's product stays below bit 16).  `bb` holds the byte in bytes 0 and 2.  (A packed
// 16-bit multiply, v_pk_mul_lo_u16, needs no mask but measured slower here: 843 against 777 us for bits 3-5 of 3.3 GB.)
__device__ __forceinline__ uint32_t step_pair(uint32_t x, uint32_t bb) {
    return __umul24((x ^ bb) & 0x00FF00FFu, kPrimeLow);
}
// A segment's words as its passes read them: word k of half A and word k of half B become one word of their bytes 0
// and 1 and one of their bytes 2 and 3, [a0 a1 b0 b1] and [a2 a3 b2 b3].  The bytes of an even step then lie in bytes 0
// and 2 of a word, where the machines' states are, and those of an odd step one shift by 8 away: one operation per four
// bytes in each pass, where picking the two bytes of every step out of the plain words took two.
__device__ __forceinline__ uint32_t low_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
// Its own inverse on the pairs: plain words to step words and back.
__device__ __forceinline__ void pair_words(uint32_t (&w)[kFnvLaneBytes / 4]) {
#pragma unroll
    for (int k = 0; k < kHalfWords; ++k) {
        const uint32_t a = w[k], b = w[kHalfWords + k];
        w[k] = low_halves(a, b);
        w[kHalfWords + k] = high_halves(a, b);
    }
}

// Makes the words new to the compiler: it would otherwise compute each word's shift once and keep it, 64 more registers,
// from one pass to the next (68 spilled words).
__device__ __forceinline__ void renew_words(uint32_t (&w)[kFnvLaneBytes / 4]) {
#pragma unroll
    for (int k = 0; k < kFnvLaneBytes / 4; ++k) asm volatile("" : "+v"(w[k]));
}

// ---- the sum on the matrix cores (what it computes and its weights: sc_hash_math.hpp) ----------------------------------
__device__ const SumWeights g_sum_weights = sum_weights();
constexpr int kWeightChunks = int(sizeof(SumWeights) / 16);
__constant__ LanePow kLanePow = lane_pow();

using i32x4 = __attribute__((ext_vector_type(4))) int32_t;
// The sum over a wave's whole segments, relative to the end of the wave's last segment, spread over its lanes (their
// values add up to it).  `w`: the step words; `m`: the true low byte at the segment's start in the low half and at its
// midpoint in the high half.  Every lane of the wave takes part: one without a whole segment passes zeros in both,
// whose products the correction cancels.
__device__ __forceinline__ uint64_t wave_sum(const uint32_t (&w)[kFnvLaneBytes / 4], uint32_t m, int lane,
                                             const u32x4* weights) {
    const uint32_t start = m & 0xFFu;
    i32x4 even = {0, 0, 0, 0}, odd = {0, 0, 0, 0};
#pragma unroll
    for (int pair = 0; pair < kHalfWords / 2; ++pair) {
        const u32x4 b = weights[pair * 64 + lane];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int k = 2 * pair + half;
            u32x4 a;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t word = i < 2 ? w[k] : w[kHalfWords + k];
                m = step_pair(m, (i & 1) ? word >> 8 : word);
                a[i] = m ^ 0x80808080u;
            }
            const i32x4 av = __builtin_bit_cast(i32x4, a), bv = __builtin_bit_cast(i32x4, b);
            if (half == 0) even = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, even, 0, 0, 0);
            else odd = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, odd, 0, 0, 0);
        }
    }
    const i32x4 s = (lane & 8) ? odd : even;
    constexpr uint64_t p1 = prime_pow_of(kFnvLaneBytes), p2 = p1 * p1, p3 = p2 * p1;
    const uint64_t rows = times_pow<p3>(s.x) + times_pow<p2>(s.y) + times_pow<p1>(s.z) + uint64_t(int64_t(s.w));
    const uint64_t ends = uint64_t((m >> 16) & 0xFFu) - times_pow<p1>(int32_t(start)) + kOffsetSum;
    return rows * kLanePow.col[lane] + ends * kLanePow.v[lane];
}

// One step of the full hash given the true low byte `l` of the state: accumulate d = (l ^ b) - l, then multiply.
__device__ __forceinline__ void step_full(uint32_t b, uint32_t& l, uint64_t& acc) {
    const uint32_t x = (l ^ b) & 0xFFu;
    acc = (acc + uint64_t(int64_t(int32_t(x) - int32_t(l)))) * kFnvPrime;
    l = __umul24(x, kPrimeLow) & 0xFFu;
}

// The same map of a partial or unaligned segment (whole segments run from registers, below), a byte at a time from
// memory; `low` holds the true bits below kJ at the segment's start.
template <int kJ, int kBits>
__device__ __forceinline__ uint32_t map_bytes(const uint8_t* p, uint32_t n, uint32_t low) {
    uint32_t e[1 << (kBits - 2)], par = 0;
#pragma unroll
    for (uint32_t m = 0; m < (1u << (kBits - 2)); ++m) e[m] = low | (m << kJ);
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t b = p[i];
        par ^= b;
#pragma unroll
        for (uint32_t& x : e) x = __umul24((x ^ b) & 0xFFu, kPrimeLow);
    }
    return map_of<kJ, kBits>(e, par, n & 1u);
}

// The maps of a wave's lanes, lane after lane.  A bit at a lane is the wave's start bit xor the parity of the terms of the
// lanes before it, and each lane's term is picked by its own true lower bits: a ballot, a count of the lower lanes (mbcnt)
// and a shift per term, on the vector units (as 64-bit scalar xor prefixes, 12 dependent operations each, the same took
// twice the instructions on the path that every later workgroup waits for).
__device__ __forceinline__ uint32_t lower_parity(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u)) & 1u;
}
__device__ __forceinline__ uint32_t parity(uint64_t mask) { return uint32_t(__popcll(mask)) & 1u; }
__device__ __forceinline__ uint64_t ballot_bit(uint32_t v) { return __ballot((v & 1u) != 0u); }
// The wave's map.  `at` are the wave's start bits before bit kBit, `lane_at` what they are at the lane.
template <int kBits, int kBit = 0>
__device__ __forceinline__ uint32_t wave_map(uint32_t lane_map, uint32_t at = 0, uint32_t lane_at = 0) {
    constexpr uint32_t base = (1u << kBit) - 1u;
    const uint64_t t = ballot_bit(lane_map >> (base + lane_at));
    uint32_t m = parity(t) << (base + at);
    if constexpr (kBit + 1 < kBits) {
        const uint32_t p = lower_parity(t);
        m |= wave_map<kBits, kBit + 1>(lane_map, 2u * at, 2u * lane_at + p) |
             wave_map<kBits, kBit + 1>(lane_map, 2u * at + 1u, 2u * lane_at + (p ^ 1u));
    }
    return m;
}
// Through the wave from its start state `st`: its end state, and this lane's start state in `at_lane`.
template <int kBits>
__device__ __forceinline__ uint32_t wave_apply(uint32_t lane_map, uint32_t st, uint32_t& at_lane) {
    uint32_t end = st, at = 0;
    at_lane = 0;
#pragma unroll
    for (int i = 0; i < kBits; ++i) {
        const uint64_t t = ballot_bit(lane_map >> ((1u << i) - 1u + at));
        const uint32_t bit = lower_parity(t) ^ ((st >> i) & 1u);
        end ^= parity(t) << i;
        at_lane |= bit << i;
        at = 2u * at + bit;
    }
    return end;
}

// The state the hash starts from: the launch's seed, or the running hash at `seed_dev` when the input continues an
// earlier one (read by every kernel that needs it, so one stream can chain pieces without a host round trip).
__device__ __forceinline__ uint64_t start_state(uint64_t seed, const uint64_t* seed_dev) {
    return seed_dev ? *seed_dev : seed;
}

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
    const uint32_t lo = __shfl_xor(uint32_t(v), m), hi = __shfl_xor(uint32_t(v >> 32), m);
    return (uint64_t(hi) << 32) | lo;
}

// One partial or unaligned segment's Horner sum, scaled by p^(bytes after it), from the true low byte `l` at its
// start, a byte at a time.
__device__ __forceinline__ uint64_t segment_sum(const uint8_t* p, uint64_t n, uint64_t begin, uint32_t l) {
    const uint64_t len = n - begin < kFnvLaneBytes ? n - begin : kFnvLaneBytes;
    uint64_t acc = 0;
    for (uint64_t i = 0; i < len; ++i) step_full(p[i], l, acc);
    return acc * pow_prime(n - begin - len);
}

__constant__ FinishPow kFinishPow = finish_pow();

// Closes a hash, one wave: h = seed * p^n + the sums of the workgroups (mod 2^64; the order of the additions does not
// matter), continued over the `tail_len` bytes at `tail` (the last partial lane segment of an aligned input, under 256
// bytes).  `ctl` holds the launch's sums and its fault word (null for an empty input): a wait that ran out (kFaultWait) or
// carries that do not match the input (kFaultCarry) make h unusable, and the launch says so at `fault_out` - the fault
// word, 0 for none, or, for a chained piece (`sticky`), or'ed into what the earlier pieces left there, so a chain reports
// a fault of any of its pieces.  With `verdict`, also 1 there when h equals `expected` and the launch has no fault, else
// 0: a later kernel on the stream can act on the check without a host round trip.
// What bounds it is its chain of dependent operations, which every hash waits for: the powers are a product over the lanes,
// one bit of the exponent each, and the tail is hashed as the lane segments are, four bytes a lane in two levels (one
// thread doing both took 5-8 us, and a tail hashed by its lane in the one-pass kernel, a byte load at a time, longer).
__global__ void __launch_bounds__(64) fnv_finish_kernel(const uint32_t* ctl, uint64_t seed, const uint64_t* seed_dev, uint64_t n,
                                                        uint64_t* out, uint32_t* fault_out, bool sticky, uint64_t expected,
                                                        uint32_t* verdict, const uint8_t* tail, uint32_t tail_len) {
    const uint32_t lane = threadIdx.x;
    // this lane's bytes of the tail
    const uint32_t count = tail_len > 4u * lane ? min(tail_len - 4u * lane, 4u) : 0u;
    uint32_t bytes[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) bytes[i] = i < count ? tail[4u * lane + i] : 0u;
    const uint64_t* acc = reinterpret_cast<const uint64_t*>(ctl + 2);
    const uint64_t start = start_state(seed, seed_dev), whole = ctl ? acc[0] : 0u, part = ctl ? acc[1] : 0u;
    const uint32_t bad = ctl ? ctl[1] : 0u;   // kFaultWait and / or kFaultCarry
    // the whole segments' sums are relative to the end of the last 64 KiB
    const uint32_t past = uint32_t((kFnvGroupBytes - n % kFnvGroupBytes) % kFnvGroupBytes);
    uint64_t pow_n = (n >> lane) & 1u ? kFinishPow.square[lane] : 1u;
    uint64_t back = lane < 16u && ((past >> lane) & 1u) ? kFinishPow.back[lane] : 1u;
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) pow_n *= shfl_xor64(pow_n, m), back *= shfl_xor64(back, m);
    uint64_t h = start * pow_n + whole * back + part;
    if (tail_len) {
        uint32_t low = 0;   // the true low byte at the lane's bytes, level by level
        const auto level = [&](auto first_bit) {
            constexpr int kJ = decltype(first_bit)::value;
            uint32_t e[4], par = 0, at;
#pragma unroll
            for (uint32_t m = 0; m < 4; ++m) e[m] = low | (m << kJ);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                par ^= bytes[i];
#pragma unroll
                for (uint32_t& x : e)
                    if (i < count) x = __umul24((x ^ bytes[i]) & 0xFFu, kPrimeLow);
            }
            const uint32_t map = count ? map_of<kJ, 4>(e, par, count & 1u) : 0u;
            (void) wave_apply<4>(map, (uint32_t(h) >> kJ) & 15u, at);
            low |= at << kJ;
        };
        level(std::integral_constant<int, 0>{});
        level(std::integral_constant<int, 4>{});
        uint64_t sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (i < count) step_full(bytes[i], low, sum);
        sum *= kFinishPow.small[count ? tail_len - 4u * lane - count : 0u];
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) sum += shfl_xor64(sum, m);
        h = h * kFinishPow.small[tail_len] + sum;
    }
    if (lane != 0) return;
    out[0] = h;
    if (fault_out) fault_out[0] = sticky ? (fault_out[0] | bad) : bad;
    if (verdict) verdict[0] = h == expected && !bad ? 1u : 0u;
}

// ---- the one-pass hash ---------------------------------------------------------------------------------------------
// One kernel reads the input once: each lane keeps its 256-byte segment in registers through the levels of the low byte
// and the sums.  A level's workgroup start state comes from a decoupled look-back rather than a scan kernel: workgroups
// take their index from a ticket counter in the order they start, publish their map of the level's state as soon as they
// have it and their end state once they know their start, and a workgroup finds its start by reading the words of the 64
// workgroups before it at once and composing maps back to the nearest end state.  A workgroup waits only on lower tickets,
// held by workgroups that are running or done, so every wait ends; each wait is also bounded (kSpinLimit reads), after
// which the launch records a fault that fails the verdict and the workgroup publishes an end state anyway, so no other
// workgroup waits on it.
// The lane within its wave, from the exec-independent lane count (two VALU operations): used where keeping threadIdx.x
// live across the kernel would spill it and reload it from scratch, a memory round trip each time.
__device__ __forceinline__ int lane_id() { return int(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u))); }
// Sleeps of 64 x 64 cycles before a look-back's first read of its window (the mapped kernel's last level writes its
// gathered payload instead): 3.3 GB hashed in 1.344 ms with two, 1.369 with one, and 0.48 GB in 249 us with two, 253 with
// three (3.3 GB alike)
constexpr int kFirstSleeps = 2, kFirstSleepsMapped = 0;
constexpr uint32_t kSpinLimit = 1u << 16;   // reads of one window, about 0.2 s (sc_fnv1a64_set_spin_limit)
// A bound the host sets only to test failure handling: every look-back of a workgroup after the first runs out at
// once, so any input of more than one workgroup (64 KiB) ends with the fault set, deterministically.
constexpr uint32_t kForceFault = 0xFFFFFFFFu;

// The launch's fault word: 0, or the or of kFaultWait (a look-back wait ran out) and kFaultCarry (a workgroup of a check
// given carries did not end with the carry after it: the input or its carries are not what was hashed).
constexpr uint32_t kFaultWait = SC_FNV_FAULT_WAIT, kFaultCarry = SC_FNV_FAULT_CARRY;
__device__ __forceinline__ void flag_fault(uint32_t* fault, uint32_t v) {
    __hip_atomic_fetch_or(fault, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish(uint32_t* status, uint32_t v) {
    __hip_atomic_store(status, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t peek(const uint32_t* status) {
    return __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The one-pass kernel's arguments.  They are read where they are needed, through the argument segment with scalar loads
// (kernel_args: a pointer that is new to the compiler each time): held in scalar registers across the kernel they pushed
// its wave masks out of them (70-95 spilled scalars).
template <int v>
using Int = std::integral_constant<int, v>;
struct OnepassArgs {
    const uint8_t* data;        // the input (16-byte aligned: `aligned`), or null with `map`
    uint64_t n;                 // bytes hashed in the kernel: an aligned input's whole lane segments
    uint64_t seed;
    const uint64_t* seed_dev;
    uint32_t* ctl;              // [0] the ticket counter, [1] the fault word, [2..3], [4..5] the sums of whole and of partial segments
    uint32_t* status;           // [workgroup][level], kStatusWords each
    HashMapArgs map;
    FnvCarries carries;
    uint64_t carry_count;
    uint32_t groups;            // workgroups' worth of input (64 KiB each), the tail that the closing kernel hashes included
    uint32_t pieces;            // 64 KiB pieces of the n bytes hashed in the kernel
    uint32_t spin_limit;
    uint32_t aligned;
};
using ConstArgs = const __attribute__((address_space(4))) OnepassArgs;
__device__ __forceinline__ ConstArgs* kernel_args() {
    ConstArgs* p = (ConstArgs*) __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}
// Where the payload's segments put payload byte 0 of workgroup g's 64 KiB, which lie in one of them: `base` + o addresses
// payload byte o.
__device__ __forceinline__ uint8_t* payload_base(uint32_t g) {
    ConstArgs* a = kernel_args();
    const uint32_t k = uint32_t((uint64_t(__umulhi(g, a->map.seg_div.m)) + g) >> a->map.seg_div.s);
    return a->map.seg[k] - uint64_t(k) * a->map.seg_bytes;
}
// The low byte the hash starts from.
__device__ __forceinline__ uint32_t start_byte() {
    ConstArgs* a = kernel_args();
    return uint32_t(start_state(a->seed, a->seed_dev)) & 0xFFu;
}

// A workgroup's status word of one level: 0, kHasMap | map or kHasState | state.
constexpr uint32_t kHasMap = 1u << 16, kHasState = 1u << 17;
// The levels of a hash that looks back: two of four bits.  Each costs 7-10 us from a workgroup's map to its start bits (see
// fnv_onepass_kernel), more than the machines a third level saves (13.5 vector operations per two bytes with three levels of
// 3, 3 and 2 bits, 17 with two): 3.3 GB in 1.36 against 1.41 ms, the 128K capture and hash in 1.76 against 1.89 ms.  A check given carries never waits
// and takes the three levels: 0.87 against 1.02 ms.
constexpr uint32_t kStatusWords = 2;

// Workgroup g's start state at one level, run by one whole wave (the result is wave-uniform); the caller has published
// g's map, and its end state is published after.  Lane l reads the status word of workgroup top - 64 + l; before workgroup
// 0 stands the start state.  The maps after the nearest end state compose like those of a wave's lanes, so resolving a
// window costs the same wherever that state lies.  Reading 128 or 256 words at once measured slower (on a
// form of the kernel that hashed 3.3 GB in 1.60 ms, 1.66 and 1.87: every read of a line that other XCDs write costs them all).
template <int kLevel, int kJ, int kBits>
__device__ __forceinline__ uint32_t look_back(uint32_t g, uint32_t map, int first_sleeps) {
    const int lane = lane_id();
    uint32_t* const status = kernel_args()->status + kLevel;
    const auto settle = [&](uint32_t st) {
        if (lane == 0) publish(status + g * kStatusWords, kHasState | apply<kBits>(map, st));
        return st;
    };
    const auto fault = [&] {   // successors still get an end state
        if (lane == 0) flag_fault(kernel_args()->ctl + 1, kFaultWait);
        return settle(0u);
    };
    const uint32_t init = g < 64u ? (start_byte() >> kJ) & state_mask<kBits>() : 0u;
    if (g == 0) return settle(init);
    const uint32_t spin_limit = kernel_args()->spin_limit;
    if (spin_limit == kForceFault) return fault();   // the failure-handling tests' forced fault (never set otherwise)
    // the workgroups just before g publish their maps about 2 us after g on average (their work varies with what shares
    // their SIMDs), so a read right away would mostly find the window incomplete and cost a round trip and a sleep anyway
    for (int i = 0; i < first_sleeps; ++i) __builtin_amdgcn_s_sleep(64);
    uint32_t acc = 0;   // the maps of the workgroups from `top` up to g, composed
    uint32_t spins = 0;
    for (int32_t top = int32_t(g);;) {
        const int32_t h = top - 64 + lane;
        const uint32_t word = h >= 0 ? peek(status + uint32_t(h) * kStatusWords) : (kHasState | init);
        const uint64_t have_state = __ballot((word & kHasState) != 0u), ready = __ballot(word != 0u);
        const int at = have_state ? 63 - __builtin_clzll(have_state) : -1;   // the lane of the nearest end state
        const uint64_t need = at == 63 ? 0u : ~0ull << (at + 1);
        if ((ready & need) != need) {   // a workgroup between that end state and g has not published its map yet
            if (++spins > spin_limit) return fault();   // never in a correct launch
            // a long sleep (64 x 64 cycles, about 1.7 us) leaves the SIMD's issue slots to the other waves' level work and
            // the status lines to their writers: sleeps of 8-32 measured alike for the plain hash and slower for the
            // fused one
            __builtin_amdgcn_s_sleep(64);
            continue;
        }
        const uint32_t after = lane > at ? word & map_mask<kBits>() : 0u;   // the maps after that end state
        if (at >= 0) {
            uint32_t unused;
            const uint32_t st = uint32_t(__builtin_amdgcn_readlane(int(word), at)) & state_mask<kBits>();
            return settle(apply<kBits>(acc, wave_apply<kBits>(after, st, unused)));
        }
        acc = compose<kBits>(acc, wave_map<kBits>(after));   // all maps: read the window before
        top -= 64;
        spins = 0;
    }
}

__constant__ GroupPow kGroupPow = group_pows();
__device__ __forceinline__ uint64_t group_pow(int byte, uint32_t k) { return kGroupPow.v[byte][(k >> (8 * byte)) & 255u]; }

struct LevelLds {
    uint32_t map[3][kFnvThreads / 64];   // per level, so that a level's maps are not rewritten while they are read
    uint32_t state, ticket;
    uint64_t sum[kFnvThreads / 64], part[kFnvThreads / 64];   // the waves' sums of whole and of partial segments
};

// One level, once every lane has its map of the level (`lane_map`, the identity 0 for a lane past the input): forms and
// publishes the workgroup's map, runs `during` in every wave (work that does not need the level's result, done while the
// look-back waits), looks back for the workgroup's start state after `first_sleeps` sleeps of 64 x 64 cycles, and returns
// this lane's start bits of the level (bit 0 upward); `end_bits` gathers the workgroup's end state.  Given carries
// (`before` is the one before the workgroup, its start state), every wave has the start state at once.
template <bool kCarried, int kLevel, int kJ, int kBits, typename During>
__device__ __forceinline__ uint32_t resolve_level(int wave, uint32_t lane_map, uint32_t g, LevelLds& L, int first_sleeps,
                                                  During during, uint32_t before, uint32_t& end_bits) {
    const int lane = lane_id();
    const uint32_t own = wave_map<kBits>(lane_map);
    if (lane == 0) L.map[kLevel][wave] = own;
    __syncthreads();
    // the waves' maps, lane k holding wave k's, compose as a wave's lanes do
    const uint32_t waves = lane < kFnvThreads / 64 ? L.map[kLevel][lane] : 0u;
    uint32_t st;
    if constexpr (kCarried) {
        during();
        st = (before >> kJ) & state_mask<kBits>();
    } else {
        uint32_t sum = 0;
        if (wave == 0) {
            sum = wave_map<kBits>(waves);
            if (lane == 0 && g > 0) publish(kernel_args()->status + g * kStatusWords + kLevel, kHasMap | sum);
        }
        during();
        if (wave == 0) {
            st = look_back<kLevel, kJ, kBits>(g, sum, first_sleeps);
            if (lane == 0) L.state = st;
        }
        __syncthreads();
        st = __builtin_amdgcn_readfirstlane(L.state);
    }
    uint32_t at_wave, bits;
    end_bits |= wave_apply<kBits>(waves, st, at_wave) << kJ;
    (void) wave_apply<kBits>(lane_map, uint32_t(__builtin_amdgcn_readlane(int(at_wave), wave)), bits);
    return bits;
}

// The levels of a whole segment held in registers, run as its two halves of kPairBytes bytes side by side (half A the
// first, half B the second): half A's map of the level in the low 16 bits and half B's above.  `w` holds the step words
// (pair_words), `par` the xor of half A's bytes in byte 0 and of half B's in byte 2, `low` the true bits
// below the level at half A's start in byte 0 and at half B's in byte 2.
__device__ __forceinline__ uint32_t half_parities(const uint32_t (&w)[kFnvLaneBytes / 4]) {
    uint32_t z = 0;
#pragma unroll
    for (int k = 0; k < kFnvLaneBytes / 4; ++k) z ^= w[k];
    return (z ^ (z >> 8)) & 0x00FF00FFu;
}
template <int kJ, int kBits>
__device__ __forceinline__ uint32_t level_maps(const uint32_t (&w)[kFnvLaneBytes / 4], uint32_t low, uint32_t par) {
    constexpr int kMachines = 1 << (kBits - 2);
    uint32_t a[kMachines], b[kMachines];
    if constexpr (kJ == 0) {
        // the lowest bits follow l' = 3 (l ^ b) mod 2^kBits (179 = 3 mod 16): a machine takes one byte of a register
        // (three times a 4-bit state stays below 2^8, and the next step masks what is above the state), half A's from
        // bit 0 = 0 and 1 in bytes 0 and 1, half B's in bytes 2 and 3, register m from m in the bits above
        static_assert(kBits == 3 || kBits == 4, "the machines' products stay in their bytes");
        constexpr uint32_t kMask = state_mask<kBits>() * 0x01010101u;
        uint32_t x[kMachines / 2];
#pragma unroll
        for (uint32_t m = 0; m < kMachines / 2; ++m) x[m] = 2u * m * 0x01010101u + 0x01000100u;
#pragma unroll
        for (int k = 0; k < kHalfWords; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t word = i < 2 ? w[k] : w[kHalfWords + k];
                const uint32_t b4 = __builtin_amdgcn_perm(word, word, (i & 1) ? 0x03030101u : 0x02020000u);
#pragma unroll
                for (uint32_t& m : x) {
                    const uint32_t y = (m ^ b4) & kMask;
                    m = y + (y << 1);
                }
            }
#pragma unroll
        for (int m = 0; m < kMachines; ++m) {
            a[m] = x[m >> 1] >> (8 * (m & 1));
            b[m] = x[m >> 1] >> (16 + 8 * (m & 1));
        }
    } else {
        // two machines a register, half A's in byte 0 and half B's in byte 2, register m from m in the level's lowest bits
#pragma unroll
        for (uint32_t m = 0; m < kMachines; ++m) a[m] = low | ((m << kJ) * 0x00010001u);
#pragma unroll
        for (int k = 0; k < kHalfWords; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t word = i < 2 ? w[k] : w[kHalfWords + k], bb = (i & 1) ? word >> 8 : word;
#pragma unroll
                for (uint32_t& m : a) m = step_pair(m, bb);
            }
#pragma unroll
        for (int m = 0; m < kMachines; ++m) b[m] = a[m] >> 16;
    }
    return map_of<kJ, kBits>(a, par, 0u) | (map_of<kJ, kBits>(b, par >> 16, 0u) << 16);
}

// ---- the gather fused with the hash -------------------------------------------------------------------------------
// A lane of the mapped hash gathers its segment of the payload from the extents' sources into its registers, stores it
// into the payload and hashes it from the registers, so a capture's payload is written and hashed in one read of the
// slot.  Most segments lie inside one extent and one contiguous source (a 256-byte segment of a 4 KiB page); the
// others, at extent and page boundaries, take their chunks one at a time.
__device__ __forceinline__ void put16(uint8_t* p, u32x4 v) { *(gu32x4*) p = v; }

// A run of the payload from payload offset `o`: bytes [o, end) come from one contiguous source `src` (a copy extent, a
// page of a pages extent, the payload itself for a self extent or an unplaced page) or are zeros (src null); `store`
// says whether the gather writes them (self bytes stay as the payload holds them).
struct Run {
    const uint8_t* src;
    uint64_t end;
    bool store;
};
__device__ __forceinline__ Run run_at(const HashExtent& x, uint64_t o, uint8_t* dst_o) {
    Run r{dst_o, x.end, false};
    if (x.kind == kExtCopy) {
        r.src = x.src + (o - x.off);
        r.store = true;
    } else if (x.kind == kExtZero) {
        r.src = nullptr;
        r.store = true;
    } else if (x.kind == kExtPages) {
        const uint32_t q = uint32_t((o - x.off) >> 4), page = q / x.page_chunks, ch = q - page * x.page_chunks;
        const uint64_t page_end = x.off + (uint64_t(page) + 1u) * x.page_chunks * 16u;
        r.end = page_end < x.end ? page_end : x.end;
        const int64_t phys = x.table ? int64_t(x.table[page]) : int64_t(page);
        if (phys >= 0 && phys < x.ld) {
            r.src = x.src + (uint64_t(phys) * x.page_chunks + ch) * 16u;
            r.store = true;
        }
    }
    return r;
}

// Read for zero runs and by lanes past the payload's whole segments, so that every lane takes the same loads.
__device__ u32x4 g_hash_zeros[kFnvLaneBytes / 16];

// Where a lane's segment is gathered from: chunk k at (k < ka ? a : b) + 16 k.  Every kind of extent comes down to one or
// two contiguous runs, and the loads stand once, after them: with loads of their own in each branch the 64 registers they
// meet in did not line up, and every path stored a chunk to scratch and read it back before the first level.
struct SegmentSource {
    const uint8_t* a;
    const uint8_t* b;
    uint32_t ka;
};
__device__ __forceinline__ const uint8_t* zero_run() { return reinterpret_cast<const uint8_t*>(g_hash_zeros); }
__device__ __forceinline__ SegmentSource one_run(const uint8_t* p) { return {p, p, kFnvLaneBytes / 16}; }
__device__ __forceinline__ SegmentSource two_runs(const Run& a, const Run& b, uint32_t ka) {
    return {a.src ? a.src : zero_run(), (b.src ? b.src : zero_run()) - 16u * ka, ka};
}
__device__ __forceinline__ void load_source(const SegmentSource& f, uint32_t (&w)[kFnvLaneBytes / 4]) {
#pragma unroll
    for (int k = 0; k < kFnvLaneBytes / 16; ++k) {
        const u32x4 v = *(const gu32x4*) ((uint32_t(k) < f.ka ? f.a : f.b) + 16 * k);
        w[4 * k] = v.x;
        w[4 * k + 1] = v.y;
        w[4 * k + 2] = v.z;
        w[4 * k + 3] = v.w;
    }
}

// A lane's whole segment inside extent X, where X holds the lane's whole wave and is wave-uniform (its fields stay in
// scalar registers and no lane reads the extent table): a copy, the payload's own bytes or zeros in one run, pages in one
// run or two (across one page boundary).  False for a segment over three pages or more (pages under 256 bytes), which the
// caller gathers chunk by chunk.
__device__ __forceinline__ bool gather_in_extent(const HashExtent& X, uint8_t* base, uint64_t begin, SegmentSource& from) {
    if (X.kind != kExtPages) {
        from = one_run(X.kind == kExtCopy ? X.src + (begin - X.off) : X.kind == kExtSelf ? base + begin : zero_run());
        return true;
    }
    const uint64_t seg_end = begin + kFnvLaneBytes;
    const Run a = run_at(X, begin, base + begin);
    Run b = a;
    uint32_t ka = kFnvLaneBytes / 16;
    if (a.end < seg_end) {
        ka = uint32_t((a.end - begin) >> 4);
        b = run_at(X, a.end, base + a.end);
        if (b.end < seg_end) return false;
    }
    from = two_runs(a, b, ka);
    return true;
}

// The lane's segment [begin, begin + len), walking the extent table from the workgroup's first extent (a wave over an
// extent boundary, a workgroup over three extents or more, the payload's last wave).  A segment in one run or two is
// loaded from them; a segment over three runs or more, and the payload's last partial segment, goes chunk by chunk into
// the payload, which the lane then reads back (its own stores, after a fence).  The payload is written by store_wave
// below (the last partial segment only here; its chunks are hashed by the closing kernel).
__device__ __forceinline__ SegmentSource gather_segment(const HashExtent* ext, uint8_t* base, uint32_t e_group, uint64_t begin,
                                                        uint64_t len) {
    uint32_t e = e_group;
    while (ext[e].end <= begin) ++e;
    HashExtent x = ext[e];
    const uint64_t seg_end = begin + len;
    const Run a = run_at(x, begin, base + begin);
    if (len == kFnvLaneBytes) {
        if (a.end >= seg_end) return two_runs(a, a, kFnvLaneBytes / 16);
        const uint32_t ka = uint32_t((a.end - begin) >> 4);   // chunks from run a
        if (a.end >= x.end) x = ext[++e];
        const Run b = run_at(x, a.end, base + a.end);
        if (b.end >= seg_end) return two_runs(a, b, ka);
        // three runs or more: walk from the workgroup's first extent again (the look-ahead above may have moved past
        // the extent holding `begin`)
        e = e_group;
        while (ext[e].end <= begin) ++e;
        x = ext[e];
    }
#pragma unroll 1
    for (uint64_t o = begin; o < seg_end;) {
        while (x.end <= o) x = ext[++e];
        const Run r = run_at(x, o, base + o);
        const uint64_t o0 = o, end = r.end < seg_end ? r.end : seg_end;
        for (; o < end; o += 16)
            if (r.store) put16(base + o, r.src ? *(const gu32x4*) (r.src + (o - o0)) : u32x4{0u, 0u, 0u, 0u});
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // the lane's stores complete before its reads
    return one_run(len == kFnvLaneBytes ? base + begin : zero_run());
}

// The wave's 16 KiB of gathered payload into the payload with coalesced stores: each lane holds 256 contiguous bytes,
// so stores straight from the registers would put 64 lines under every store instruction (measured: the fused kernel
// 3.3-3.7 ms with them against 2.3 ms without any store, and 8.2 ms with non-temporal ones, in an earlier form).  Eight
// passes of 2 KiB: an eighth of the lanes write their segments' step words into the wave's LDS rows (17 chunks apart), then
// every lane reads back a chunk of step words and its partner, pairs them into a chunk of each half and stores the two: a
// store instruction writes eight runs of 128 bytes, the first or the second halves of eight segments.  Non-temporal stores:
// the 128K capture + hash 1.776 ms against 1.825 with regular ones, a paged 16381-token one 336 against 348 us.  Bytes at or
// past `limit` (the part hashed in the kernel) are not written here.
constexpr int kXposeRow = kFnvLaneBytes / 16 + 1;   // chunks per LDS row: a lane's 16 and one of padding
__device__ __forceinline__ void store_wave(u32x4 (&lds)[8 * kXposeRow], const uint32_t (&w)[kFnvLaneBytes / 4],
                                           uint8_t* dst, uint64_t wave_begin, uint64_t limit, int lane) {
#pragma unroll
    for (int pass = 0; pass < 8; ++pass) {
        if ((lane >> 3) == pass) {
            const int row = (lane & 7) * kXposeRow;
#pragma unroll
            for (int k = 0; k < kFnvLaneBytes / 16; ++k)
                lds[row + k] = u32x4{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // step words 4c .. 4c + 3 of this pass's segment lane / 8 and their partners: chunk c of each half
        const int seg = lane >> 3, c = lane & 7;
        const u32x4 lo = lds[seg * kXposeRow + c], hi = lds[seg * kXposeRow + kHalfWords / 4 + c];
        const u32x4 a = {low_halves(lo.x, hi.x), low_halves(lo.y, hi.y), low_halves(lo.z, hi.z), low_halves(lo.w, hi.w)};
        const u32x4 b = {high_halves(lo.x, hi.x), high_halves(lo.y, hi.y), high_halves(lo.z, hi.z),
                         high_halves(lo.w, hi.w)};
        const uint64_t o = wave_begin + uint64_t(pass) * 2048u + uint64_t(seg) * kFnvLaneBytes + uint64_t(c) * 16u;
        if (o < limit) {   // whole segments: both chunks
            __builtin_nontemporal_store(a, (gu32x4*) (dst + o));
            __builtin_nontemporal_store(b, (gu32x4*) (dst + o + kPairBytes));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// kMapped: the payload is gathered through `map` (stored, and hashed up to `n`, its whole lane segments) instead of read
// from `data`.  Not kMapped, with `map.seg` set: the payload is read where its segments hold it (`data` unused).
// What bounds it: its 17 vector operations per two bytes, at 82% busy vector units, and the two look-backs, 9.9 and 7.5 us of
// a workgroup's 33 from its map to its start bits (the maps' arithmetic, the wait for the latest of the workgroups before it
// and the words' way through memory).  Given carries it neither waits nor takes tickets, and the vector units are 99% busy;
// gathering, 62%, its reads and look-backs slowed by its own writes.  3.3 GB in 1.344 ms (1.76 ms with three levels and the
// sums on the vector units), checked with carries in 0.87-0.88 (1.29), the 128K slot gathered and hashed in 1.776 (2.03).
// Five waves per SIMD (96 VGPRs).  Taking several 64 KiB per workgroup, as the carried check does, measured slower here (3.3
// GB in 1.60 ms): the workgroups' starts then spread over 3-5 us instead of 2, and every look-back waits for the latest.
template <bool kMapped, bool kCarried>
__global__ void __launch_bounds__(kFnvThreads) __attribute__((amdgpu_waves_per_eu(5, 8))) fnv_onepass_kernel(OnepassArgs) {
    __shared__ LevelLds L;
    __shared__ u32x4 s_xpose[kMapped ? kFnvThreads / 64 : 1][8 * kXposeRow];
    __shared__ u32x4 s_weights[kWeightChunks];
    if (!kCarried && threadIdx.x == 0) L.ticket = atomicAdd(kernel_args()->ctl, 1u);
    // the sums' weights into LDS, by `threads` threads
    const auto stage_weights = [&](uint32_t thread, uint32_t threads) {
#pragma unroll 2
        for (uint32_t i = thread; i < uint32_t(kWeightChunks); i += threads)
            s_weights[i] = ((const gu32x4*) &g_sum_weights.w[0][0][0])[i];
    };
    if constexpr (kCarried) stage_weights(threadIdx.x, kFnvThreads);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // mapped: the table of extents, and the end of the last extent of the lane's share of it
    const HashExtent* ext = nullptr;
    uint32_t n_ext = 0;
    uint64_t share_end = 0;
    if constexpr (kMapped) {
        ConstArgs* a = kernel_args();
        ext = a->map.ext, n_ext = a->map.n_ext;
        share_end = ext[ExtentSpan{0u, n_ext}.sample(threadIdx.x % 64u)].end;
    }
    __syncthreads();
    uint64_t total = 0, total_part = 0;   // thread 0: the workgroup's sums
    uint32_t g = kCarried ? blockIdx.x : __builtin_amdgcn_readfirstlane(L.ticket);
#pragma unroll 1
    do {
        const int lane = lane_id();
        // the lane's segment: its first byte, and whether it is whole (and aligned), partial or past the input.  The
        // mapped instance hashes whole lane segments only (its launch passes n rounded down to them, the closing kernel
        // takes the rest), so the byte-at-a-time forms drop out of it
        const auto begin_of = [&] { return ((uint64_t(g) * kFnvThreads + uint32_t(wave) * 64u) + uint32_t(lane)) * kFnvLaneBytes; };
        const auto bytes_of = [&] {
            const uint64_t begin = begin_of(), n = kernel_args()->n;
            return begin >= n ? 0u : n - begin < kFnvLaneBytes ? uint32_t(n - begin) : uint32_t(kFnvLaneBytes);
        };
        const auto address_of = [&]() -> const uint8_t* {
            ConstArgs* a = kernel_args();
            const uint64_t begin = begin_of();
            return (a->map.seg ? payload_base(g) : a->data) + begin;
        };
        const uint32_t len = bytes_of();
        const bool full = kMapped ? len != 0u : len == kFnvLaneBytes && kernel_args()->aligned;
        const bool bytes = !kMapped && !full && len != 0u;
        // a check's carries around this workgroup
        uint32_t before = 0, after = 0;
        if constexpr (kCarried) {
            ConstArgs* a = kernel_args();
            before = g > 0 ? uint32_t(a->carries.in[g - 1]) : start_byte();
            after = g < a->carry_count ? uint32_t(a->carries.in[g]) : 0x100u;
        }
        // what the workgroup's sum is worth where the last one ends; read here, with the data, rather than when the sum is
        // there and everything else done (mapped: once the loads' sources are found, which these reads would hold up: the
        // 128K capture + hash 1.776 against 1.789 ms; the plain hash the other way, 1.344 against 1.348)
        uint64_t worth = 0;
        const auto read_worth = [&] {
            const uint32_t rest = kernel_args()->pieces - 1u - g;   // (the tail's own workgroup sums nothing)
            worth = group_pow(0, rest) * group_pow(1, rest) * group_pow(2, rest) * group_pow(3, rest);
        };
        if constexpr (!kMapped) read_worth();
        uint32_t w[kFnvLaneBytes / 4] = {};
        uint8_t* base = nullptr;   // mapped: `base` + o addresses payload byte o in the segment holding this workgroup's bytes
        if constexpr (kMapped) {
            // the extent holding the workgroup's first byte: every lane has read the end of the last extent of its share of
            // the table while the ticket was on its way; a table of more than 64 is sampled again inside the share found
            ConstArgs* a = kernel_args();
            const uint64_t lo = uint64_t(g) * kFnvGroupBytes;
            ExtentSpan span{0u, n_ext};
            span.narrow(uint32_t(__popcll(__ballot(share_end <= lo))));
            while (span.size > 1u) span.narrow(uint32_t(__popcll(__ballot(ext[span.sample(uint32_t(lane))].end <= lo))));
            const uint32_t first = span.first;
            // that extent and the next, read together through the constant address space (scalar loads; the map does not
            // change during the launch, and consecutive workgroups read the same lines) and held from here
            typedef const __attribute__((address_space(4))) uint64_t ConstWord;
            const ConstWord* q0 = (const ConstWord*) (ext + first);
            const ConstWord* q1 = (const ConstWord*) (ext + min(first + 1u, n_ext - 1u));
            uint64_t h[12];
#pragma unroll
            for (int i = 0; i < 6; ++i) h[i] = q0[i], h[6 + i] = q1[i];
            base = payload_base(g);
            asm volatile("" ::"s"(h[0]), "s"(h[1]), "s"(h[2]), "s"(h[3]), "s"(h[4]), "s"(h[5]), "s"(h[6]), "s"(h[7]),
                         "s"(h[8]), "s"(h[9]), "s"(h[10]), "s"(h[11]));
            HashExtent x0, x1;
            static_assert(sizeof(HashExtent) == 48, "the words read are the extent's fields");
            __builtin_memcpy(&x0, h, 48);
            __builtin_memcpy(&x1, h + 6, 48);
            const uint64_t begin = begin_of(), n_total = a->map.n_total;
            SegmentSource from = one_run(zero_run());
            if (begin < n_total) {
                const uint64_t wave_lo = (uint64_t(g) * kFnvThreads + uint64_t(wave) * 64) * kFnvLaneBytes;
                const uint64_t wave_hi = wave_lo + 64u * kFnvLaneBytes;
                bool done = false;
                if (wave_hi <= n_total) {   // every lane of the wave whole, inside one of the two extents
                    if (wave_hi <= x0.end)
                        done = gather_in_extent(x0, base, begin, from);
                    else if (wave_lo >= x0.end && wave_hi <= x1.end)
                        done = gather_in_extent(x1, base, begin, from);
                }
                if (!done) {
                    const uint64_t left = n_total - begin;
                    from = gather_segment(ext, base, first, begin, left < kFnvLaneBytes ? left : kFnvLaneBytes);
                }
            }
            load_source(from, w);
        } else if (full) {
            load_segment(address_of(), w);
        }
        if constexpr (kMapped) read_worth();
        // every load is issued before the first word is used: paired as they come, the first two loads' words had the others
        // wait for a memory round trip
        __builtin_amdgcn_sched_barrier(0);
        pair_words(w);

        // the levels: every lane's map of the level (a whole segment from its two halves in registers, a partial or unaligned
        // one a byte at a time), then the workgroup's start state.  `s` gathers the true start bits at the lane's segment,
        // `sb` at its midpoint (its first half's map applied to the level's start bits)
        const uint32_t par = full ? half_parities(w) : 0u;
        uint32_t s = 0, sb = 0, end_bits = 0;   // end_bits: the workgroup's end state, level by level (its carry)
        const auto level = [&](auto index, auto first_bit, auto width, int first_sleeps, auto during) {
            constexpr int kLevel = decltype(index)::value, kJ = decltype(first_bit)::value, kBits = decltype(width)::value;
            uint32_t halves = 0, lane_map = 0;
            if constexpr (kLevel > 0) renew_words(w);
            if (full) {
                halves = level_maps<kJ, kBits>(w, s | (sb << 16), par);
                lane_map = compose<kBits>(halves >> 16, halves & map_mask<kBits>());
            } else if (bytes) {
                lane_map = map_bytes<kJ, kBits>(address_of(), bytes_of(), s);
            }
            const uint32_t st = resolve_level<kCarried, kLevel, kJ, kBits>(wave, lane_map, g, L, first_sleeps, during, before,
                                                                           end_bits);
            s |= st << kJ;
            sb |= apply<kBits>(halves & map_mask<kBits>(), st) << kJ;
        };
        if constexpr (kCarried) {
            level(Int<0>{}, Int<0>{}, Int<3>{}, 0, [] {});
            level(Int<1>{}, Int<3>{}, Int<3>{}, 0, [] {});
            level(Int<2>{}, Int<6>{}, Int<2>{}, 0, [] {});
        } else {
            // the waves that do not look back stage the weights meanwhile: before the ticket they spread the workgroups'
            // starts, which every look-back then waits for
            level(Int<0>{}, Int<0>{}, Int<4>{}, kFirstSleeps, [&] {
                if (wave > 0) stage_weights(uint32_t(wave - 1) * 64u + uint32_t(lane), kFnvThreads - 64u);
            });
            // the gathered payload is written while the last look-back waits (stores issued earlier meet the next
            // workgroups' gathers, later ones hold up the workgroup's end)
            level(Int<1>{}, Int<4>{}, Int<4>{}, kMapped ? kFirstSleepsMapped : kFirstSleeps, [&] {
                if constexpr (kMapped) {
                    store_wave(s_xpose[wave], w, base, (uint64_t(g) * kFnvThreads + uint64_t(wave) * 64) * kFnvLaneBytes,
                               kernel_args()->n, lane);
                }
            });
        }
        if (wave == 0 && lane == 0) {
            ConstArgs* a = kernel_args();
            if (a->carries.out && g < a->carry_count) a->carries.out[g] = uint8_t(end_bits);
            if (kCarried && after != 0x100u && end_bits != after) flag_fault(a->ctl + 1, kFaultCarry);
        }

        // the sums, from the true low bytes at the segment's start and midpoint: the wave's whole segments together
        // (relative to the end of its last segment), a partial or unaligned one a byte at a time
        renew_words(w);
        uint64_t acc = 0;
        if (__ballot(full)) acc = wave_sum(w, full ? s | (sb << 16) : 0u, lane, s_weights);
        for (int m = 32; m > 0; m >>= 1) acc += shfl_xor64(acc, m);
        uint64_t part = 0;
        if (!kMapped && __ballot(bytes)) {
            if (bytes) part = segment_sum(address_of(), kernel_args()->n, begin_of(), s);
            for (int m = 32; m > 0; m >>= 1) part += shfl_xor64(part, m);
        }
        if (lane == 0) {
            L.sum[wave] = acc;
            L.part[wave] = part;
        }
        __syncthreads();
        if (wave == 0 && lane == 0) {
            constexpr uint64_t wave_pow = prime_pow_of(64u * kFnvLaneBytes);
            uint64_t sum = 0, parts = 0;
#pragma unroll
            for (int q = 0; q < kFnvThreads / 64; ++q) {
                sum = sum * wave_pow + L.sum[q];
                parts += L.part[q];
            }
            total += sum * worth;
            total_part += parts;
        }
        g += gridDim.x;
    } while (kCarried && g < kernel_args()->groups);
    if (threadIdx.x == 0) {
        uint32_t* ctl = kernel_args()->ctl;
        atomicAdd(reinterpret_cast<unsigned long long*>(ctl + 2), (unsigned long long) total);
        if (total_part) atomicAdd(reinterpret_cast<unsigned long long*>(ctl + 4), (unsigned long long) total_part);
    }
}

// Clears the status words, the ticket and fault words and the sum before a launch (a kernel rather than a memset, so a
// graph may hold it).
__global__ void __launch_bounds__(kThreads) fnv_onepass_init_kernel(uint32_t* status, uint64_t words, uint32_t* ctl) {
    const uint64_t stride = uint64_t(gridDim.x) * kThreads;
    for (uint64_t i = uint64_t(blockIdx.x) * kThreads + threadIdx.x; i < words; i += stride) status[i] = 0u;
    if (blockIdx.x == 0 && threadIdx.x < 6) ctl[threadIdx.x] = 0u;
}
}  // namespace

// The bound on each look-back wait, in window reads; tests lower it to force a wait to run out.
std::atomic<uint32_t> g_spin_limit{kSpinLimit};

// Workspace: [ticket, fault and sum words][status words: kStatusWords per workgroup].
FnvWorkspace fnv_workspace(uint64_t n) {
    FnvWorkspace w{};
    w.segments = (n + kFnvLaneBytes - 1) / kFnvLaneBytes;
    w.groups = (w.segments + kFnvThreads - 1) / kFnvThreads;
    auto up = [](uint64_t x) { return (x + 255) / 256 * 256; };
    w.off_ctl = 0;
    w.off_status = 256;
    w.bytes = w.off_status + up(kStatusWords * 4 * w.groups);
    return w;
}

// Clears a launch's words and enqueues the one-pass kernel over `a` (its ctl, status, groups, pieces and spin limit set
// here); returns ctl, or null for an empty input, which needs neither.
template <bool kMapped>
uint32_t* enqueue_onepass(OnepassArgs a, uint8_t* workspace, uint64_t bytes, hipStream_t stream) {
    const FnvWorkspace w = fnv_workspace(bytes);
    if (!w.groups) return nullptr;
    a.ctl = reinterpret_cast<uint32_t*>(workspace + w.off_ctl);
    a.status = reinterpret_cast<uint32_t*>(workspace + w.off_status);
    a.groups = uint32_t(w.groups);
    a.pieces = uint32_t(fnv_workspace(a.n).groups);
    a.spin_limit = g_spin_limit.load();
    const uint64_t words = kStatusWords * w.groups, init_blocks = (words + kThreads - 1) / kThreads < 1024 ? (words + kThreads - 1) / kThreads : 1024;
    hipLaunchKernelGGL(fnv_onepass_init_kernel, dim3(unsigned(init_blocks)), dim3(kThreads), 0, stream, a.status, words, a.ctl);
    if (!kMapped && a.carries.in) {
        // no workgroup waits for another: each takes up to four 64 KiB in turn, which spares it the start of a workgroup
        // (3.3 GB checked in 0.884 ms against 0.907 with one each and 0.895 with eight) while others' kernels still get
        // their turn on the CUs; fewer when that would leave some of the 1280 (five per CU) without work.  Between a few
        // rounds of 1280 it costs the last round's idle CUs: 0.48 GB, 1838 workgroups of four, 155 us against 143 with one
        // each
        const uint32_t turns = a.groups < 2 * 1280 ? 1 : a.groups < 4 * 1280 ? a.groups / 1280 : 4;
        hipLaunchKernelGGL((fnv_onepass_kernel<false, true>), dim3((a.groups + turns - 1) / turns), dim3(kFnvThreads), 0, stream, a);
    } else {
        hipLaunchKernelGGL((fnv_onepass_kernel<kMapped, false>), dim3(a.groups), dim3(kFnvThreads), 0, stream, a);
    }
    return a.ctl;
}

hipError_t launch_fnv1a64(const void* data, uint64_t n, uint64_t seed, const uint64_t* seed_dev, uint64_t* out,
                          uint32_t* fault_out, void* workspace, hipStream_t stream, uint64_t expected, uint32_t* verdict,
                          const FnvCarries& carries) {
    OnepassArgs a{};
    a.data = static_cast<const uint8_t*>(data);
    a.aligned = (reinterpret_cast<uintptr_t>(data) & 15u) == 0;
    a.n = a.aligned ? n & ~uint64_t(kFnvLaneBytes - 1) : n;
    a.seed = seed;
    a.seed_dev = seed_dev;
    a.carries = carries;
    a.carry_count = fnv_carry_count(n);
    const uint32_t* ctl = enqueue_onepass<false>(a, static_cast<uint8_t*>(workspace), n, stream);
    // the finish reads the start state before it writes `out`, so `out` may be `seed_dev` itself
    hipLaunchKernelGGL(fnv_finish_kernel, dim3(1), dim3(64), 0, stream, ctl, seed, seed_dev, a.n, out, fault_out,
                       seed_dev != nullptr, expected, verdict, a.data + a.n, uint32_t(n - a.n));
    return hipGetLastError();
}

// The gather fused with the hash: the payload's `map.n_total` bytes gathered into its segments and hashed, the whole
// lane segments in the one-pass kernel and the last partial one (under 256 bytes, at `tail`) by the closing kernel,
// which runs after every byte is in place.  A map that only reads is hashed by the plain kernel where its segments hold it.
// With `verdict`, the closing kernel also leaves the check of the hash
// against `expected` there, as sc_fnv1a64_check_async does.  The carries are those of the whole payload (`n_total`
// bytes): a carry at a boundary inside the last partial lane segment cannot occur (boundaries are 64 KiB apart).
hipError_t launch_fnv1a64_mapped(const HashMapArgs& map, const uint8_t* tail, uint64_t seed, uint64_t* out,
                                 uint32_t* fault_out, void* workspace, hipStream_t stream, uint64_t expected,
                                 uint32_t* verdict, const FnvCarries& carries) {
    const uint64_t n_total = map.n_total, n_full = n_total & ~uint64_t(kFnvLaneBytes - 1);
    if (n_total % 16) return hipErrorInvalidValue;   // maps hold whole 16-byte chunks (the closing kernel loads them)
    OnepassArgs a{};
    a.aligned = 1u;
    a.seed = seed;
    a.map = map;
    a.carries = carries;
    a.carry_count = fnv_carry_count(n_total);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    a.n = n_full;
    const uint32_t* ctl = map.store ? enqueue_onepass<true>(a, ws, n_total, stream) : enqueue_onepass<false>(a, ws, n_total, stream);
    hipLaunchKernelGGL(fnv_finish_kernel, dim3(1), dim3(64), 0, stream, ctl, seed, nullptr, n_full, out, fault_out, false,
                       expected, verdict, tail, uint32_t(n_total - n_full));
    return hipGetLastError();
}

}  // namespace sc

// ---- the hash that allocates nothing ----------------------------------------------------------------------------------
// For callers that cannot allocate (code under HIP graph capture, tight serving loops): the workspace is `scratch`, one
// array per GPU that the library holds until the process ends, sized for inputs of up to SC_FNV_NOALLOC_MAX_BYTES
// (fnv_workspace(4 GiB) is 0.5 MiB).  Every call clears all of it that it uses (the ticket, the fault word, the sum
// and the look-back's status words) with a kernel of its own before the hash kernel; a call after another on the same
// stream is ordered after it, and calls that overlap on one GPU (on different streams) race on the one array.
namespace {

constexpr uint64_t kScratchBytes = 2ull << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};   // the device address of `scratch` on each GPU, looked up once per GPU

// The current device's copy of `scratch`.  In host code the array's name is only a stand-in for the device symbol, so
// kernels get the address the runtime reports for it, looked up with the device current.
hipError_t scratch_of_current_device(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

}  // namespace

extern "C" int sc_fnv1a64_noalloc_async(const void* data, uint64_t bytes, uint64_t seed, uint64_t* out, uint32_t* fault,
                                        void* stream) {
    if (!out || !fault || (bytes && !data))
        return sc::record_error(SC_EINVAL, "sc_handoff: missing hash input, output or fault word");
    if (reinterpret_cast<uintptr_t>(fault) & 3u)
        return sc::record_error(SC_EINVAL, "sc_handoff: the hash fault word must be 4-byte aligned");
    if (bytes > SC_FNV_NOALLOC_MAX_BYTES || sc::fnv_workspace(bytes).bytes > kScratchBytes)
        return sc::record_error(SC_ERANGE, "sc_handoff: the hash without allocation takes at most 4 GiB "
                                           "(SC_FNV_NOALLOC_MAX_BYTES); use sc_fnv1a64_async with a workspace");
    void* ws = nullptr;
    hipError_t e = scratch_of_current_device(&ws);
    if (e != hipSuccess)
        return sc::record_error(SC_EHIP, std::string("sc_handoff hash scratch: ") + hipGetErrorString(e));
    e = sc::launch_fnv1a64(data, bytes, seed, nullptr, out, fault, ws, static_cast<hipStream_t>(stream), 0, nullptr,
                           sc::FnvCarries{});
    if (e != hipSuccess) return sc::record_error(SC_EHIP, std::string("sc_handoff hash launch: ") + hipGetErrorString(e));
    return sc::record_ok();
}

extern "C" int sc_fnv1a64_set_spin_limit(uint32_t reads) {
    static_assert(sc::kForceFault == SC_FNV_FORCE_FAULT, "the forced-fault bound is the header's");
    sc::g_spin_limit.store(reads ? reads : sc::kSpinLimit);
    return sc::record_ok();
}
