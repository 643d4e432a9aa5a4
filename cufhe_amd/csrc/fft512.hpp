// Folded negacyclic FP64 transform for N = 1024 (H = 512) out of six-FMA
// butterflies: the transform of the lvl1 key-bundle rotation.
//
// The 512 folded values are a polynomial modulo X^512 - i. A radix-2 step
// splits modulo X^2n - s^2 into X^n - s and X^n + s: lo = u + s v, hi = u - s v
// with one root s per block (the recursion of Longa and Naehrig's merged
// negacyclic NTT, over the complex numbers), so there is no separate twist.
// With s = c (1 + i t), t = tan, c = cos (the ratio form of Linzer and Feig,
// "Implementation of efficient FFT algorithms on fused multiply-add
// architectures", 1993):
//   p + i q = (1 + i t) v: two FMAs;  u +- c (p + i q): four FMAs
// i.e. 6 FP64 instructions a butterfly, 216 a lane and transform, against
// about 295 of the radix-8 form (fft_wave.hpp) with its twist, twiddle and
// constant multiplications. No root here has c = 0; where c is small, t is
// large and the rounding error of p, q (relative) is scaled back by c, so the
// error of a butterfly stays at that of a complex product.
// The inverse runs the steps backwards, u = lo + hi, v = conj(s) (lo - hi),
// keeping v / c and multiplying by the products of c once per three levels
// (the last three levels' products go into the caller's rounding scale).
//
// Levels 1-3 act on the eight registers (element lane + 64 r), 4-6 and 7-9
// after LDS transposes: octet o of the lanes takes block rev3(o) (so that its
// root's angle, and its place in the spectrum, grow with o). On exit lane
// c + 8 o, register a holds the value at exp(i pi (1 + 4 n) / 1024), n = o +
// 8 rev3(c) + 64 rev3(a): bin k = -n mod 512 of the engine's storage order
// (bin k = q + 8 c + 64 d at d * 64 + c + 8 q), which Slots gives. Every LDS
// access pattern puts the 16 lanes of a group on 16 different bank quads.
#pragma once

#include "fft_wave.hpp"

namespace cufhe_amd {
namespace fft512 {

constexpr int kH = 512;

// One block's roots: s of the first level, of the second, of the third and of
// the third's upper half (the third's times exp(i pi / 4)). c and t as above.
struct Root {
    double c, t;
};
struct Roots {
    Root r1, r2, r3, r3h;
    // for the inverse's scales: r3h.c / r3.c = cos(pi / 4) (1 - t3), and c2 c3
    __host__ __device__ __forceinline__ constexpr double k() const
    {
        return 0.70710678118654752440 - 0.70710678118654752440 * r3.t;
    }
    __host__ __device__ __forceinline__ constexpr double c23() const { return r2.c * r3.c; }
};
constexpr int kRootWords = 4;  // 16-byte words of a Roots
// Table layout, 16-byte words: word w of block b of a level group of B blocks
// at w * B + b. Group 1 (levels 4-6): 8 blocks (octet); group 2: 64 (lane).
constexpr int kTab1 = kRootWords * 8, kTab2 = kRootWords * 64;
constexpr int kTabWords = kTab1 + kTab2;

template <int B>
__host__ __device__ __forceinline__ Roots load_roots(const cplx* tab, int b)
{
    const cplx w0 = lds_load(&tab[b]), w1 = lds_load(&tab[B + b]), w2 = lds_load(&tab[2 * B + b]),
               w3 = lds_load(&tab[3 * B + b]);
    return Roots{{w0.x, w0.y}, {w1.x, w1.y}, {w2.x, w2.y}, {w3.x, w3.y}};
}

// Roots of levels 1-3: angles pi/4, pi/8, pi/16 and 5 pi/16.
__host__ __device__ __forceinline__ constexpr Roots first_roots()
{
    constexpr double c2 = 0.92387953251128675613, c3 = 0.98078528040323044913,
                     c3h = 0.55557023301960222474;
    return Roots{{0.70710678118654752440, 1.0},
                 {c2, 0.41421356237309504880},
                 {c3, 0.19891236737965800691},
                 {c3h, 1.49660576266548901760}};
}

// lo = u + s v, hi = u - s v (in place u, v); QUARTER: the root is i s.
template <bool QUARTER>
__host__ __device__ __forceinline__ void bfly(cplx& u, cplx& v, Root s)
{
    const double p = fma(-s.t, v.y, v.x), q = fma(s.t, v.x, v.y);
    const cplx u0 = u;
    if constexpr (!QUARTER) {
        u = cplx{fma(s.c, p, u0.x), fma(s.c, q, u0.y)};
        v = cplx{fma(-s.c, p, u0.x), fma(-s.c, q, u0.y)};
    }
    else {
        u = cplx{fma(-s.c, q, u0.x), fma(s.c, p, u0.y)};
        v = cplx{fma(s.c, q, u0.x), fma(-s.c, p, u0.y)};
    }
}
// Three forward levels on eight registers.
__host__ __device__ __forceinline__ void levels(cplx (&x)[8], const Roots& s)
{
#pragma unroll
    for (int i = 0; i < 4; i++) bfly<false>(x[i], x[i + 4], s.r1);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        bfly<false>(x[i], x[i + 2], s.r2);
        bfly<true>(x[4 + i], x[6 + i], s.r2);
    }
    bfly<false>(x[0], x[1], s.r3);
    bfly<true>(x[2], x[3], s.r3);
    bfly<false>(x[4], x[5], s.r3h);
    bfly<true>(x[6], x[7], s.r3h);
}

// u = lo + hi, v = conj(s) (lo - hi) / c; QUARTER: the root is i s.
template <bool QUARTER>
__host__ __device__ __forceinline__ void ibfly(cplx& lo, cplx& hi, double t)
{
    const cplx d = csub(lo, hi);
    lo = cadd(lo, hi);
    if constexpr (!QUARTER)
        hi = cplx{fma(t, d.y, d.x), fma(-t, d.x, d.y)};
    else
        hi = cplx{fma(-t, d.x, d.y), fma(-t, d.y, -d.x)};
}
// The same with hi in units of k times lo's.
__host__ __device__ __forceinline__ void ibfly_scaled(cplx& lo, cplx& hi, double t, double k)
{
    const cplx d = {fma(-k, hi.x, lo.x), fma(-k, hi.y, lo.y)};
    lo = cplx{fma(k, hi.x, lo.x), fma(k, hi.y, lo.y)};
    hi = cplx{fma(t, d.y, d.x), fma(-t, d.x, d.y)};
}
// Three inverse levels; register r is left in units of scale(r): the
// products of c1 (bit 2 of r), c2 (bit 1) and c3 (bit 0).
__host__ __device__ __forceinline__ void ilevels(cplx (&x)[8], const Roots& s)
{
    ibfly<false>(x[0], x[1], s.r3.t);
    ibfly<true>(x[2], x[3], s.r3.t);
    ibfly<false>(x[4], x[5], s.r3h.t);
    ibfly<true>(x[6], x[7], s.r3h.t);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        ibfly<false>(x[i], x[i + 2], s.r2.t);
        ibfly<true>(x[4 + i], x[6 + i], s.r2.t);
    }
    ibfly<false>(x[0], x[4], s.r1.t);
    ibfly_scaled(x[1], x[5], s.r1.t, s.k());
    ibfly<false>(x[2], x[6], s.r1.t);
    ibfly_scaled(x[3], x[7], s.r1.t, s.k());
}
__host__ __device__ __forceinline__ constexpr double scale(const Roots& s, int r)
{
    const double low = (r & 3) == 0 ? 1.0 : (r & 3) == 1 ? s.r3.c : (r & 3) == 2 ? s.r2.c : s.c23();
    return r & 4 ? s.r1.c * low : low;
}
__host__ __device__ __forceinline__ void rescale(cplx (&x)[8], const Roots& s)
{
#pragma unroll
    for (int r = 1; r < 8; r++) x[r] = cscale(x[r], scale(s, r));
}

// Where register a of a lane's spectrum lives in the storage order, as two
// element offsets from (7 - rev3(a)) * 64: lane 0 is a row further on, its
// register 0 wraps to row 0.
struct Slots {
    int first, rest;
    __host__ __device__ __forceinline__ static Slots of(int lane)
    {
        auto rev3 = [](int v) { return ((v & 1) << 2) | (v & 2) | (v >> 2); };
        const int n0 = lane >> 3, n1 = rev3(lane & 7);
        const int q = (8 - n0) & 7, c = (8 - n1 - (n0 != 0)) & 7;
        const int l = c + 8 * q;
        return Slots{l - (lane == 0 ? 7 * 64 : 0), l + (lane == 0 ? 64 : 0)};
    }
    __host__ __device__ __forceinline__ int at(int a) const
    {
        const int rev = ((a & 1) << 2) | (a & 2) | (a >> 2);
        return (a == 0 ? first : rest) + (7 - rev) * 64;
    }
};

// Transpose slots in a buffer of kScratch elements. First: row r (register) of
// 64, the upper four rows half a bank sweep on; octet o reads row rev3(o).
// Second, within an octet: 8 x 8 with sub-rows of 9.
constexpr int kScratch = 576;
__host__ __device__ __forceinline__ constexpr int row1(int r) { return r * 64 + 8 * (r >> 2); }
__host__ __device__ __forceinline__ int octet_row1(int lane)
{
    const int o = lane >> 3;
    return row1(((o & 1) << 2) | (o & 2) | (o >> 2)) + (lane & 7);
}
__host__ __device__ __forceinline__ int sub_a(int lane) { return (lane >> 3) * 72 + (lane & 7); }      // + 9 c
__host__ __device__ __forceinline__ int sub_b(int lane) { return (lane >> 3) * 72 + 9 * (lane & 7); }  // + a

// Forward transforms of M polynomials held by one wave (x[p][r]: folded value
// lane + 64 r), each through a buffer of its own that receives its spectrum in
// storage order. Their LDS traffic and arithmetic interleave. hook(0), (1),
// (2): called after each of the three register stages' stores.
template <int M, bool PRIO, class Hook>
__device__ __forceinline__ void forward(cplx (&x)[M][8], cplx* const (&buf)[M], const cplx* tab,
                                        const Slots& slots, int lane, Hook&& hook)
{
    wave_prio<PRIO>(3);
#pragma unroll
    for (int p = 0; p < M; p++) {
        levels(x[p], first_roots());
#pragma unroll
        for (int r = 0; r < 8; r++) lds_store(&buf[p][row1(r) + lane], x[p][r]);
    }
    hook(0);
    wave_lds_sync();
    const Roots s1 = load_roots<8>(tab, lane >> 3);
#pragma unroll
    for (int p = 0; p < M; p++)
#pragma unroll
        for (int b = 0; b < 8; b++) x[p][b] = lds_load(&buf[p][octet_row1(lane) + 8 * b]);
    wave_lds_sync();
    wave_prio<PRIO>(2);
#pragma unroll
    for (int p = 0; p < M; p++) {
        levels(x[p], s1);
#pragma unroll
        for (int c = 0; c < 8; c++) lds_store(&buf[p][sub_a(lane) + 9 * c], x[p][c]);
    }
    hook(1);
    wave_lds_sync();
    const Roots s2 = load_roots<64>(tab + kTab1, lane);
#pragma unroll
    for (int p = 0; p < M; p++)
#pragma unroll
        for (int a = 0; a < 8; a++) x[p][a] = lds_load(&buf[p][sub_b(lane) + a]);
    wave_lds_sync();
    wave_prio<PRIO>(1);
#pragma unroll
    for (int p = 0; p < M; p++) {
        levels(x[p], s2);
#pragma unroll
        for (int a = 0; a < 8; a++) lds_store(&buf[p][slots.at(a)], x[p][a]);
    }
    hook(2);
    wave_prio<PRIO>(0);
}

// Inverse transform of the spectrum in buf (storage order; the buffer is the
// scratch). x[r]: 512 times the folded value lane + 64 r, in units of
// scale(first_roots(), r).
template <bool PRIO>
__device__ __forceinline__ void inverse(cplx (&x)[8], cplx* buf, const cplx* tab, const Slots& slots,
                                        int lane)
{
#pragma unroll
    for (int a = 0; a < 8; a++) x[a] = lds_load(&buf[slots.at(a)]);
    wave_prio<PRIO>(3);
    const Roots s2 = load_roots<64>(tab + kTab1, lane);
    wave_lds_sync();
    ilevels(x, s2);
    rescale(x, s2);
#pragma unroll
    for (int a = 0; a < 8; a++) lds_store(&buf[sub_b(lane) + a], x[a]);
    wave_lds_sync();
    const Roots s1 = load_roots<8>(tab, lane >> 3);
#pragma unroll
    for (int c = 0; c < 8; c++) x[c] = lds_load(&buf[sub_a(lane) + 9 * c]);
    wave_lds_sync();
    wave_prio<PRIO>(2);
    ilevels(x, s1);
    rescale(x, s1);
#pragma unroll
    for (int b = 0; b < 8; b++) lds_store(&buf[octet_row1(lane) + 8 * b], x[b]);
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 8; r++) x[r] = lds_load(&buf[row1(r) + lane]);
    wave_lds_sync();
    wave_prio<PRIO>(1);
    ilevels(x, first_roots());
    wave_prio<PRIO>(0);
}

}  // namespace fft512
}  // namespace cufhe_amd
