// Host tables of the folded FP64 transforms (fft_wave.hpp, fft512.hpp).
#pragma once

#include <cmath>
#include <vector>

#include "fft512.hpp"

namespace cufhe_amd {

// exp(i*pi*t/N) for t in [0, 2N), computed in long double.
inline std::vector<cplx> e2n_table(int N)
{
    std::vector<cplx> e(2 * N);
    const long double pi = 3.141592653589793238462643383279502884L;
    for (int t = 0; t < 2 * N; t++) {
        const long double a = pi * static_cast<long double>(t) / static_cast<long double>(N);
        e[t] = cplx{static_cast<double>(cosl(a)), static_cast<double>(sinl(a))};
    }
    // exact values on the axes
    e[0] = {1.0, 0.0};
    e[N / 2] = {0.0, 1.0};
    e[N] = {-1.0, 0.0};
    e[3 * N / 2] = {0.0, -1.0};
    // Each root is the FP64 product of e[64 (t >> 6)] and e[t & 63], rounded as
    // the device's cmul rounds it: the words of lvl2 results depend on these
    // values. Entries t < 64 and t = 64u are unchanged.
    std::vector<cplx> p(2 * N);
    for (int t = 0; t < 2 * N; t++) {
        const cplx a = e[64 * (t >> 6)], b = e[t & 63];
        p[t] = cplx{std::fma(a.x, b.x, -a.y * b.y), std::fma(a.x, b.y, a.y * b.x)};
    }
    return p;
}

// fft512.hpp's root tables: per block of angle theta (the roots of X^n -
// exp(i theta)) cos and tan of theta / 2, / 4, / 8 and / 8 + pi / 4.
inline std::vector<cplx> fft512_tables()
{
    std::vector<cplx> t(fft512::kTabWords);
    auto fill = [&](cplx* out, int blocks, auto n_of) {
        for (int b = 0; b < blocks; b++) {
            // theta = pi / (2 blocks) * (1 + 4 n): 8 blocks after three levels, 64 after six
            const long double pi = 3.14159265358979323846264338327950288L;
            const long double theta = pi * (1 + 4 * n_of(b)) / (2 * blocks);
            const long double ang[4] = {theta / 2, theta / 4, theta / 8, theta / 8 + pi / 4};
            for (int w = 0; w < 4; w++)
                out[w * blocks + b] = cplx{static_cast<double>(cosl(ang[w])), static_cast<double>(tanl(ang[w]))};
        }
    };
    auto rev3 = [](int v) { return ((v & 1) << 2) | (v & 2) | (v >> 2); };
    fill(t.data(), 8, [&](int o) { return o; });
    fill(t.data() + fft512::kTab1, 64, [&](int l) { return (l >> 3) + 8 * rev3(l & 7); });
    return t;
}

// FFTTables' arrays for polynomials of N coefficients.
struct FoldedTables {
    std::vector<cplx> e2n, twl, tw64, cr, tws;
    explicit FoldedTables(int N) : e2n(e2n_table(N)), twl(N / 2), tw64(64), cr(N / 128), tws(64)
    {
        auto at = [&](long long t) { return e2n[static_cast<size_t>(((t % (2 * N)) + 2 * N) % (2 * N))]; };
        // twl[k2*64+l] = exp(i*pi*l/N) * exp(-2*pi*i*l*k2/H) = E[l*(1 - 4*k2)]
        for (int k2 = 0; k2 < N / 128; k2++)
            for (int l = 0; l < 64; l++) twl[k2 * 64 + l] = at(static_cast<long long>(l) * (1 - 4 * k2));
        // tw64[c*8+a] = exp(-2*pi*i*a*c/64) = E[-(2N/64)*a*c]
        for (int c = 0; c < 8; c++)
            for (int a = 0; a < 8; a++) tw64[c * 8 + a] = at(-static_cast<long long>(2 * N / 64) * a * c);
        // tws[l] = exp(-2*pi*i*l/H) = E[-4 l]
        for (int l = 0; l < 64; l++) tws[l] = at(-4LL * l);
        // cr[r] = exp(i*pi*64*r/N) = E[64 r]
        for (int r = 0; r < N / 128; r++) cr[r] = at(64LL * r);
    }
};

}  // namespace cufhe_amd
