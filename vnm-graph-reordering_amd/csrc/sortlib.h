// Device-wide sort/scan/select primitives used by the VENOM, packing and
// proposer passes (hand-written in sortlib.hip).  Scratch is per host thread
// and kernels run on `st`.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vnm_internal.h"

namespace vnm {

// The bits of a 64-bit key that a sort compares: w0 bits from s0 on, and (w1 >
// 0, then w0 < 64) w1 more significant ones from s1 on.  Bits in neither range may
// hold anything; they move with the key.
struct KeyBits {
    int s0, w0, s1, w1;
};
inline KeyBits key_range(int begin, int end) { return KeyBits{begin, end - begin, 0, 0}; }
// (hi, lo) keys of two 32-bit halves, the low half below 2^lo, the high half below 2^hi
inline KeyBits key_halves(int lo, int hi) { return KeyBits{0, lo, 32, hi}; }
// Bits that hold 0 .. x.
inline int bits_for(int64_t x) {
    int b = 1;
    while ((1ll << b) <= x) ++b;
    return b;
}

// The sorted bits of a key as one number: w0 bits from s0 on, then (w1 > 0) the
// bits from s1 on (and whatever lies above them).
__host__ __device__ __forceinline__ uint64_t sort_bits(const KeyBits &b, uint64_t k) {
    uint64_t c = k >> b.s0;
    if (b.w1) c = (c & ((1ull << b.w0) - 1)) | ((k >> b.s1) << b.w0);
    return c;
}

// One pass's digit.
struct Digit {
    KeyBits b;
    int shift, bits;
    __host__ __device__ __forceinline__ int of(uint64_t k) const { return (int)((sort_bits(b, k) >> shift) & ((1u << bits) - 1u)); }
};

// A sort's passes, and the digit's width of the one that begins at `shift` of
// `total` bits.
inline int passes_of(const KeyBits &b) { return (b.w0 + b.w1 + 7) / 8; }
__host__ __device__ inline int digit_bits(int total, int shift) {
    const int left = total - shift;
    return (left + (left + 7) / 8 - 1) / ((left + 7) / 8);
}

// Stable LSD radix sort on those bits (the input is not written; out must not
// alias it).
int sort_keys_u64(const uint64_t *in, uint64_t *out, int64_t n, KeyBits bits, hipStream_t st);
// sort_keys_u64 whose kernels all return at once while *skip is nonzero
// (read on the device when they run: a launch chain enqueued ahead of the
// decision)
int sort_keys_u64_if(const uint64_t *in, uint64_t *out, int64_t n, KeyBits bits, hipStream_t st, const int *skip);
// Grow this host thread's current scratch slot to what a sort of n keys
// (with values) needs, so that sorts up to that size allocate nothing (as
// under capture).
int sort_scratch_reserve(int64_t n);
// Make scratch slot `slot` (0..15) of this host thread the current one;
// returns the previous slot.  Sorts enqueued on streams that may run
// concurrently need separate slots.
int sort_scratch_slot(int slot);
int sort_pairs_u64_i32(const uint64_t *kin, uint64_t *kout, const int32_t *vin, int32_t *vout,
                       int64_t n, KeyBits bits, hipStream_t st);
int scan_excl_i32(const int32_t *in, int32_t *out, int64_t n, hipStream_t st);
int scan_incl_max_i32(const int32_t *in, int32_t *out, int64_t n, hipStream_t st);
// out[j] = in[i] for the j-th i with flags[i] != 0, in order; *d_count = j's.
int select_flagged_i32(const int32_t *in, const uint8_t *flags, int32_t *out, int32_t *d_count,
                       int64_t n, hipStream_t st);

}  // namespace vnm
