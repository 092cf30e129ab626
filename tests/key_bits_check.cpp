// Host check of the radix sort's digits (csrc/sortlib.h): the passes over one or two
// ranges of a key's bits, each a stable sort by its digit, order the keys as one
// stable sort by those ranges, whatever the other bits hold.  Prints "ok".
#include <hip/hip_runtime.h>

#include "sortlib.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

using namespace vnm;

static uint64_t low(int w) { return w >= 64 ? ~0ull : (1ull << w) - 1; }

int main() {
    std::mt19937_64 rng(11);
    for (int it = 0; it < 20000; ++it) {
        KeyBits b;
        if (it % 3 == 0) {
            const int w = 1 + (int)(rng() % 64), s = (int)(rng() % (65 - w));
            b = key_range(s, s + w);
        } else if (it % 3 == 1) {
            b = key_halves(1 + (int)(rng() % 32), 1 + (int)(rng() % 32));
        } else {  // two ranges anywhere, the second above the first
            const int w0 = 1 + (int)(rng() % 40), s0 = (int)(rng() % (63 - w0));
            const int s1 = s0 + w0 + (int)(rng() % (64 - s0 - w0)), w1 = 1 + (int)(rng() % (64 - s1));
            b = KeyBits{s0, w0, s1, w1};
        }
        const uint64_t few = it & 1 ? ~0ull : rng() & rng();  // many ties, or few
        std::vector<uint64_t> k(60);
        for (auto &x : k) x = rng() & few;
        auto want = k;
        std::stable_sort(want.begin(), want.end(), [&](uint64_t x, uint64_t y) {
            const uint64_t hx = b.w1 ? (x >> b.s1) & low(b.w1) : 0, hy = b.w1 ? (y >> b.s1) & low(b.w1) : 0;
            if (hx != hy) return hx < hy;
            return ((x >> b.s0) & low(b.w0)) < ((y >> b.s0) & low(b.w0));
        });
        const int total = b.w0 + b.w1;
        int shift = 0, passes = 0;
        for (; shift < total; ++passes) {
            const Digit d{b, shift, digit_bits(total, shift)};
            if (d.bits < 1 || d.bits > 8) return std::printf("a digit of %d bits\n", d.bits), 1;
            std::stable_sort(k.begin(), k.end(), [&](uint64_t x, uint64_t y) { return d.of(x) < d.of(y); });
            shift += d.bits;
        }
        if (shift != total || passes != passes_of(b)) return std::printf("%d bits in %d passes\n", shift, passes), 1;
        if (k != want) return std::printf("ranges %d+%d, %d+%d\n", b.s0, b.w0, b.s1, b.w1), 1;
    }
    for (int64_t x : {(int64_t)0, (int64_t)1, (int64_t)255, (int64_t)256, (int64_t)1 << 40})
        if (x >> bits_for(x) || (x > 1 && !(x >> (bits_for(x) - 1)))) return std::printf("bits_for\n"), 1;
    std::printf("ok\n");
    return 0;
}
