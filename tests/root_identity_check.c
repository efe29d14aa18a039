/* Checks the square root and reciprocal of the HIP pair loops (sqrt_pair and rcp_of in
 * shamrock_amd/csrc/sph.hip) against sqrt and 1 / y: seeds of 1 / sqrt(v) with relative errors up
 * to 2^-22, operands that are random, squares, near powers of two, and squares of significands of
 * all ones, exponents in [-767, 1000].  Prints the mismatches of the roots, of the reciprocals, and
 * of reciprocals by plain Newton corrections whose operand is not of all ones. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t st[2] = {0x2545f4914f6cdd1dULL, 0x9e3779b97f4a7c15ULL};
static uint64_t next(void) {
    uint64_t s1 = st[0];
    const uint64_t s0 = st[1];
    st[0] = s0;
    s1 ^= s1 << 23;
    st[1] = s1 ^ s0 ^ (s1 >> 17) ^ (s0 >> 26);
    return st[1] + s0;
}
static uint64_t bits(double d) {
    uint64_t b;
    memcpy(&b, &d, 8);
    return b;
}
static double make(int e, uint64_t m) {
    uint64_t b = ((uint64_t) (e + 1023) << 52) | (m & ((1ULL << 52) - 1));
    double d;
    memcpy(&d, &b, 8);
    return d;
}

int main(int argc, char **argv) {
    long n = argc > 1 ? atol(argv[1]) : 1000000L, bad_s = 0, bad_r = 0, other = 0, ones = 0;
    for (long i = 0; i < n; i++) {
        const uint64_t ra = next(), rb = next();
        const int e = (int) (ra % 1767) - 766, eh = (int) (ra % 800) - 380;
        double v = make(e, rb);
        switch (i & 7) {
        case 1: v = make(eh, rb) * make(eh, rb); break;
        case 2: v = make(eh, ~0ULL) * make(eh, ~0ULL); break; /* root of all ones */
        case 3: v = make(eh, ~0ULL - (rb & 0xff)) * make(eh, ~0ULL - (rb & 0xff)); break;
        case 4: v = make(eh, rb & 0xff) * make(eh, rb & 0xff); break;
        case 5: v = make(e, ~0ULL - (rb & 0xff)); break;
        case 6: v = make(e, rb & 0xff); break;
        default: break;
        }
        const double seed = (double) (int64_t) next() * 0x1p-63; /* [-1, 1) */
        const double r0   = 1.0 / sqrt(v) * (1.0 + seed * 0x1p-22);
        double s = v * r0, g = 0.5 * r0;
        const double d = fma(-g, s, 0.5);
        g = fma(g, d, g);
        s = fma(s, d, s);
        s = fma(fma(-s, s, v), g, s);
        s = fma(fma(-s, s, v), g, s);
        if (s != sqrt(v)) bad_s++;
        const double y = s;
        double r = g + g, q = r; /* q: without the turn up */
        r = fma(fma(-y, r, 1.0) + 0x1p-64, r, r);
        r = fma(fma(-y, r, 1.0), r, r);
        q = fma(fma(-y, q, 1.0), q, q);
        q = fma(fma(-y, q, 1.0), q, q);
        if (r != 1.0 / y) bad_r++;
        if (q != 1.0 / y) {
            if ((bits(y) & ((1ULL << 52) - 1)) == (1ULL << 52) - 1) ones++;
            else other++;
        }
    }
    printf("of all ones, without the turn up: %ld\n%ld %ld %ld\n", ones, bad_s, bad_r, other);
    return ones == 0; /* the exception is real */
}
