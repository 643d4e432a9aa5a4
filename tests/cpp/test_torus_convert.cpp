// double_to_torus and turns_to_torus32 on the host: rint(v) mod 2^w of doubles
// around every place where their steps change (ties, the 2^31 / 2^32 / 2^63 / 2^64
// edges, half turns, large values), against integer arithmetic on the double's
// mantissa. Runs without a GPU.
#include "../../cufhe_amd/csrc/device_common.hpp"

#include <cmath>
#include <cstdio>
#include <cstdlib>

// rint(v) mod 2^64: the mantissa shifted in 64-bit arithmetic; values below
// 2^62 through llrint (ties to even).
static uint64_t exact(double v)
{
    if (std::fabs(v) < 4611686018427387904.0) return static_cast<uint64_t>(std::llrint(v));
    int e;
    const double m = std::frexp(v, &e);  // v = m 2^e, 0.5 <= |m| < 1
    const int64_t mant = static_cast<int64_t>(std::ldexp(m, 53));
    return e - 53 >= 64 ? 0 : static_cast<uint64_t>(mant) << (e - 53);
}

static uint64_t rnd_state = 88172645463325252ull;
static uint64_t rnd()
{
    rnd_state ^= rnd_state << 13;
    rnd_state ^= rnd_state >> 7;
    rnd_state ^= rnd_state << 17;
    return rnd_state;
}

static long checked = 0;
static void check(double v)
{
    const uint64_t want = exact(v);
    const uint64_t got64 = cufhe_amd::double_to_torus<uint64_t>(v);
    if (got64 != want) {
        std::printf("Torus64 of %a: %016llx, not %016llx\n", v, (unsigned long long)got64,
                    (unsigned long long)want);
        std::exit(1);
    }
    checked++;
    // the same value given in turns (2^-32 is a power of two: no rounding)
    const uint32_t turns = cufhe_amd::turns_to_torus32(v * 0x1p-32);
    if (turns != static_cast<uint32_t>(want)) {
        std::printf("turns %a: %08x, not %08x\n", v * 0x1p-32, turns, static_cast<uint32_t>(want));
        std::exit(1);
    }
    const uint32_t got32 = cufhe_amd::double_to_torus<uint32_t>(v);
    if (got32 != static_cast<uint32_t>(want)) {
        std::printf("Torus32 of %a: %08x, not %08x\n", v, got32, static_cast<uint32_t>(want));
        std::exit(1);
    }
}

int main()
{
    for (int e = -3; e <= 100; e++) {
        const double p = std::ldexp(1.0, e);
        for (double base : {p, 1.5 * p, 3.0 * p, std::nextafter(p, 0.0), std::nextafter(p, 4 * p)})
            for (double d : {0.0, 0.25, 0.5, 0.75, 1.0, 1.5, 2147483648.0, 2147483647.5, 2147483648.5,
                             4294967296.0, 9223372036854775808.0, 18446744073709551616.0})
                for (double s : {1.0, -1.0}) {
                    check(s * (base + d));
                    check(s * (base - d));
                }
    }
    for (int i = 0; i < 2000000; i++) {
        const double m = static_cast<double>(static_cast<int64_t>(rnd())) * 0x1p-63;
        check(std::ldexp(m, static_cast<int>(rnd() % 90)));
        // halves: ties at the unit position
        check(static_cast<double>(static_cast<int64_t>(rnd()) >> (12 + rnd() % 40)) + 0.5);
    }
    std::printf("ok: %ld values\n", checked);
    return 0;
}
