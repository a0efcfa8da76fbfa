// hx::quot (csrc/physics.hpp) against the division, bit for bit: random pairs, significands at the ends of the
// binade, the quotients closest to the middle between two doubles, and its exceptions.  argv[1]: pairs.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>

#include "physics.hpp"

static uint64_t state = 0x9e3779b97f4a7c15ull;
static uint64_t rnd()
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return state;
}

static long wrong = 0, tried = 0;
static double quot(double a, double b) { return hx::quot(a, b, 1.0 / b); }
static void same(double a, double b)
{
    const double q = quot(a, b), d = a / b;
    ++tried;
    if (std::memcmp(&q, &d, sizeof(q)) && ++wrong <= 5) std::printf("%a / %a: %a, division %a\n", a, b, q, d);
}

// x with odd * x = 1 modulo m = 2^k-coprime, by the extended Euclidean algorithm
static int64_t inverse(uint64_t x, uint64_t m)
{
    __int128 r0 = (__int128)m, r1 = x % m, t0 = 0, t1 = 1;
    while (r1) {
        const __int128 q = r0 / r1, r = r0 - q * r1, t = t0 - q * t1;
        r0 = r1; r1 = r; t0 = t1; t1 = t;
    }
    return (int64_t)(t0 < 0 ? t0 + (__int128)m : t0);
}

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main(int argc, char **argv)
{
    const long n = argc > 1 ? std::atol(argv[1]) : 1000000;
    const uint64_t top = 1ull << 52, mask = top - 1;
    for (long x = 0; x < n; ++x) {
        // significands: anywhere, or within a few units of a power of two
        auto significand = [&]() {
            const uint64_t r = rnd(), near = (r >> 4) & 15;
            return top | (r & 3 ? (r >> 8) & mask : r & 4 ? near : mask - near);
        };
        const double a = std::ldexp((double)significand(), (int)(rnd() % 200) - 152), b = std::ldexp((double)significand(), (int)(rnd() % 60) - 82);
        same(rnd() & 1 ? a : -a, b);
    }
    const long random = wrong;
    // a / b = (M -+ 1/b) / 2^k with M odd and of 54 bits: a 2^k = +-1 modulo b
    for (long x = 0; x < n / 10; ++x) {
        const uint64_t b = top | (rnd() & mask) | 1;
        for (int below = 0; below < 2; ++below) {
            const int k = below ? 54 : 53;   // quotients in [1/2, 1) and in [1, 2)
            const uint64_t inv = (uint64_t)inverse((uint64_t)(((unsigned __int128)1 << k) % b), b);
            for (uint64_t a : {inv, b - inv}) {
                if (!below) a += b;
                if (below && 2 * a < b) continue;
                if (a >> 53 && a & 1) continue;   // not a double
                same((double)a, (double)b);
            }
        }
    }
    // small numerators, down to where the remainder still is a normal number or zero
    for (long x = 0; x < n / 10; ++x)
        same(std::ldexp((double)(top | (rnd() & mask)), -968 - 52), std::ldexp((double)(top | (rnd() & mask)), (int)(rnd() % 40) - 72));
    std::printf("%ld pairs, %ld wrong (%ld of the random ones)\n", tried, wrong, random);
    CHECK(wrong == 0);
    // the exceptions
    const double inf = std::numeric_limits<double>::infinity(), nan = std::nan(""), sub = 1e-310;
    CHECK(quot(0.0, 1.3) == 0.0 && quot(-0.0, 1.3) == 0.0 && !std::signbit(quot(-0.0, 1.3)));
    CHECK(std::isnan(quot(inf, 1.3)) && std::isnan(quot(-inf, 1.3)) && std::isnan(quot(1.0, inf)));
    CHECK(std::isnan(quot(1.0, 0.0)) && std::isnan(quot(0.0, 0.0)) && std::isnan(quot(1.0, sub)));
    CHECK(std::isnan(quot(nan, 1.0)) && std::isnan(quot(1.0, nan)));
    return 0;
}
