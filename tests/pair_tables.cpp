// The trit kernel's pair tables (tq1_bytes.h) over every byte value, on the
// host: indices inside their tables, legal bytes giving their digits' operand
// pairs in fp16 and bf16.
#include <stdint.h>
#include <stdio.h>

#include "tq1_bytes.h"

using namespace tq1_bytes;

static int failures = 0;
static void expect(bool ok, const char *what, unsigned a, unsigned b) {
    if (!ok && ++failures <= 20) printf("FAIL %s at %u, %u\n", what, a, b);
}

static int digit(unsigned byte, int i) {
    for (; i; --i) byte /= 3;
    return static_cast<int>(byte % 3);
}

// -1, 0 or +1 of a digit, in a 16-bit type whose 1 has the bits `one`.
static uint32_t value(int d, uint32_t one) { return d == 0 ? one | 0x8000u : (d == 2 ? one : 0u); }

int main() {
    for (unsigned p = 0; p < 256; ++p) {
        expect(kPairT27a + 2 * (p / 9) + 1 < kPairT27b, "T27a index", p, 0);
        expect(kPairT27b + 2 * (p % 27) + 1 < kPairT9a, "T27b index", p, 0);
        expect(kPairT9a + 2 * (p % 9) + 1 < kPairT9b, "T9a index", p, 0);
        expect(kPairT9b + p / 27 < kPairEntries, "T9b index", p, 0);
        expect(kPairT27b + 2 * tail_entry(p) + 1 < kPairT9a, "tail index", p, 0);
        expect((p * 57u) >> 9 == p / 9, "code byte 24's split", p, 0);
    }
    const int spans[4] = {kPairT27b - kPairT27a, kPairT9a - kPairT27b, kPairT9b - kPairT9a, kPairEntries - kPairT9b};
    for (int i = 0; i < 4; ++i) expect(spans[i] <= 64, "a table spans at most the 64 banks", i, 0);
    const uint32_t ones[2] = {0x3c00u, 0x3f80u};
    const uint32_t scaled[4] = {ones[0], ones[1], 0x3b80u, 0x3f00u};  // and bf16's 2^-8, fp32's 2^-1
    for (uint32_t one : scaled) {
        for (int i = 0; i < kPairEntries; ++i)  // every half is -1, 0 or +1, illegal bytes' too
            for (int h = 0; h < 2; ++h) {
                const uint32_t half = (pair_entry(i, one) >> (16 * h)) & 0xffffu;
                expect(half == 0 || (half & 0x7fffu) == one, "operand half", i, h);
            }
        for (unsigned a = 0; a < 243; ++a)
            for (unsigned b = 0; b < 243; ++b) {
                const int ta = kPairT27a + 2 * (a / 9), tb = kPairT27b + 2 * (b % 27);
                const uint32_t got[5] = {pair_entry(kPairT9a + 2 * (a % 9), one), pair_entry(ta, one),
                                         pair_entry(ta + 1, one) | pair_entry(tb, one), pair_entry(tb + 1, one),
                                         pair_entry(kPairT9b + b / 27, one)};
                for (int q = 0; q < 5; ++q) {
                    const int lo = 2 * q, hi = 2 * q + 1;
                    const uint32_t want = value(lo < 5 ? digit(a, lo) : digit(b, lo - 5), one) |
                                          (value(hi < 5 ? digit(a, hi) : digit(b, hi - 5), one) << 16);
                    expect(got[q] == want, "a byte pair's operands", a, b);
                }
            }
        for (unsigned p = 0; p < 243; ++p)
            for (unsigned t = 0; t < 27; ++t) {
                // dwords 30 and 31: code byte 24's first four digits; its fifth and the tail's three
                const int h = kPairT27a + 2 * (p / 9), m = kPairT27b + 2 * static_cast<int>(tail_entry(t));
                expect(pair_entry(kPairT9a + 2 * (p % 9), one) ==
                           (value(digit(p, 0), one) | (value(digit(p, 1), one) << 16)), "code byte 24, digits 0-1", p, t);
                expect(pair_entry(h, one) == (value(digit(p, 2), one) | (value(digit(p, 3), one) << 16)),
                       "code byte 24, digits 2-3", p, t);
                expect((pair_entry(h + 1, one) | pair_entry(m, one)) ==
                           (value(digit(p, 4), one) | (value(digit(t, 0), one) << 16)), "code byte 24 and tail", p, t);
                expect(pair_entry(m + 1, one) == (value(digit(t, 1), one) | (value(digit(t, 2), one) << 16)),
                       "tail digits 1-2", p, t);
            }
    }
    printf(failures ? "%d violations\n" : "ok\n", failures);
    return failures ? 1 : 0;
}
