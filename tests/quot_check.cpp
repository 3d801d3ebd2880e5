// Host check of the ray set-up's quotients (ngi_quot.h) against the IEEE
// division.  Reciprocals: every significand at 7 exponents, from both numbers
// around the reciprocal (a hardware reciprocal is one of them: within 1 ulp),
// the greatest significand from the correct one only.  Quotients: pairs over the range that quot_exact accepts, the corners
// of it among them, and numerators that make a quotient a tie of denormal
// numbers, which must be refused or divided correctly.  Prints "ok <probes>"
// and exits 0, or prints the first mismatch and exits 1.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

#include "ngi_quot.h"

using namespace ngi;

static float bits(uint32_t u) {
    float f;
    memcpy(&f, &u, 4);
    return f;
}
static uint32_t word(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    return u;
}

static long g_probes = 0;

static bool quotient(float n, float d) {
    if (std::fabs(n) > std::fabs(d) || !quot_exact(std::fabs(n), d)) return true;
    ++g_probes;
    const float q = div_markstein(n, d, 1.0f / d);
    if (word(q) == word(n / d)) return true;
    printf("%a / %a: %a, not %a\n", n, d, q, n / d);
    return false;
}

int main() {
    for (uint32_t e : {62u, 63u, 100u, 126u, 127u, 128u, 152u})   // 2^-65 (1e-20 is above 2^-67) to 2^25
        for (uint32_t m = 0; m < 1u << 23; ++m) {
            const float d = bits((m & 1u) << 31 | e << 23 | m), r = 1.0f / d;
            const double x = 1.0 / d;   // (double)r lies on the other side of it, or on it
            const float other = std::nextafter(r, std::fabs(r) < std::fabs(x) ? 2.0f * r : 0.0f);
            for (float from : {r, m == 0x7fffffu ? r : other}) {
                ++g_probes;
                if (word(rcp_newton(d, from)) != word(r)) {
                    printf("1 / %a from %a: %a\n", d, from, rcp_newton(d, from));
                    return 1;
                }
            }
        }
    std::mt19937 rng(7);
    auto number = [&](uint32_t lo, uint32_t hi) { return bits((rng() & 0x807fffffu) | (lo + rng() % (hi - lo + 1)) << 23); };
    for (int i = 0; i < 20000000; ++i)
        if (!quotient(number(26, 152), number(60, 153))) return 1;   // 2^-101 .. 2^25, 2^-67 .. 2^26
    for (int i = 0; i < 4000000; ++i) {
        // Near 2^-100 and just below 2^26: the smallest quotients.
        if (!quotient(number(27, 28), number(150, 153))) return 1;
        // Quotients that are odd multiples of 2^-150: halfway between denormal numbers.
        const uint32_t odd = 2u * (rng() % 4096u) + 1u;
        const float d = bits((rng() & 0x007ff000u) | (150u + rng() % 103u) << 23);
        if (!quotient(std::ldexp(d * (float)odd, -150), d)) return 1;
    }
    printf("ok %ld\n", g_probes);
    return 0;
}
