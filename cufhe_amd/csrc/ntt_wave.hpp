// Wavefront-level negacyclic NTT over Z_P, P = 2147473409 (N = 1024).
//
// Reference: include/ntt_small_modulus.cuh:38-74 (the prime), :154-282
// (modular ops), :394-509 (SmallForwardNTT/SmallInverseNTT, CT/GS). The
// results of the NTT backend are exact residues, so only the transform's
// mathematics must match, not its butterfly order or roots: any primitive
// 2N-th root psi gives the same negacyclic products bit for bit.
//
// Arithmetic: Montgomery multiplication with R = 2^32 (P < 2^31), operands
// canonical in [0, P). Twiddles and keys are stored in Montgomery form
// (x R mod P), data in normal form, so mont(data, twiddle) stays normal.
//
// Transform (one wave per polynomial, like fft_wave.hpp): coefficient
// i = lane + 64 r (r < 16) in VGPRs; Z[k] = sum_i x_i psi^(i (2k+1)):
// twist psi^i = psi^lane * psi^(64 r) (lane factor merged into the step-2
// twiddle), 16-point DFT over registers, twiddle, 64-point DFT over lanes as
// 8 x 8 with two LDS transposes laid out so that both access patterns of
// each transpose hit 64 distinct banks with 4-byte elements. Output: lane
// L = c + 8q, register g*8+d holds Z[k], k = (q+8g) + 16(c+8d), stored at
// p = (g*8+d)*64 + L.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#include "fft_wave.hpp"  // wave_lds_sync, static_for

namespace cufhe_amd {
namespace ntt31 {

constexpr uint32_t P = 2147473409u;  // 1048571 * 2^11 + 1
constexpr uint32_t HALF_P = P / 2;

constexpr uint64_t powmod(uint64_t b, uint64_t e)
{
    uint64_t r = 1;
    b %= P;
    while (e) {
        if (e & 1) r = r * b % P;
        b = b * b % P;
        e >>= 1;
    }
    return r;
}
// -P^-1 mod 2^32 (Newton iteration)
constexpr uint32_t neg_inv()
{
    uint32_t x = 1;
    for (int i = 0; i < 5; i++) x *= 2u - P * x;
    return 0u - x;
}
constexpr uint32_t PINV = neg_inv();
constexpr uint32_t R1 = static_cast<uint32_t>((1ULL << 32) % P);               // R mod P
constexpr uint32_t R2 = static_cast<uint32_t>((uint64_t)R1 * R1 % P);           // R^2 mod P
constexpr uint32_t to_mont_c(uint32_t x) { return static_cast<uint32_t>(((uint64_t)x << 32) % P); }

// Primitive 2N-th root of unity (N = 1024): g^((P-1)/2048) for the smallest
// quadratic non-residue g.
constexpr uint32_t find_psi()
{
    uint64_t g = 2;
    while (powmod(g, (P - 1) / 2) != P - 1) g++;
    return static_cast<uint32_t>(powmod(g, (P - 1) / 2048));
}
constexpr uint32_t PSI = find_psi();
constexpr uint32_t PSI_INV = static_cast<uint32_t>(powmod(PSI, 2047));
static_assert(powmod(PSI, 1024) == P - 1, "psi must be a primitive 2048-th root");

// root_pow(e) = psi^e (normal form), e taken mod 2048
constexpr uint32_t psi_pow(int64_t e) { return static_cast<uint32_t>(powmod(PSI, ((e % 2048) + 2048) % 2048)); }

}  // namespace ntt31

__device__ __forceinline__ uint32_t mod_add(uint32_t a, uint32_t b)
{
    const uint32_t s = a + b;  // < 2P < 2^32
    return s >= ntt31::P ? s - ntt31::P : s;
}
__device__ __forceinline__ uint32_t mod_sub(uint32_t a, uint32_t b)
{
    const uint32_t d = a - b;  // a < b: wraps above 2^31 > P, and d + P is the residue
    return __builtin_elementwise_min(d, d + ntt31::P);
}
// r mod P for r < 2P: min(r, r - P) (r - P wraps above r when r < P). Written
// as an unsigned min so it stays two VALU ops; a compare on the 64-bit
// Montgomery sum (what `r >= P ? r - P : r` folds into) costs a 64-bit
// compare, a select and a VCC hazard wait.
__device__ __forceinline__ uint32_t reduce_2p(uint32_t r)
{
    return __builtin_elementwise_min(r, r - ntt31::P);
}
// a * b * R^-1 mod P, canonical, for b < P and any 32-bit a: t + m P is below
// 2^33 P < 2^64 and its upper word below 2P. A sum a + b or a difference
// a + P - b of residues can therefore be a factor as it is.
__device__ __forceinline__ uint32_t mont_mul(uint32_t a, uint32_t b)
{
    const uint64_t t = static_cast<uint64_t>(a) * b;
    const uint32_t m = static_cast<uint32_t>(t) * ntt31::PINV;
    const uint64_t u = t + static_cast<uint64_t>(m) * ntt31::P;  // < 2^63 + 2^63
    return reduce_2p(static_cast<uint32_t>(u >> 32));            // u >> 32 < 2P
}

// (a1 b1 + a2 b2) R^-1 mod P with one Montgomery reduction: the 64-bit sum
// is below 2 P^2, so t + m P < 2^64 and the result is below 2P before the
// final subtraction. Equal to mod_add(mont_mul(a1, b1), mont_mul(a2, b2))
// for canonical inputs (every value here is a residue in [0, P)).
__device__ __forceinline__ uint32_t mont_dot2(uint32_t a1, uint32_t b1, uint32_t a2, uint32_t b2)
{
    const uint64_t t = static_cast<uint64_t>(a1) * b1 + static_cast<uint64_t>(a2) * b2;
    const uint32_t m = static_cast<uint32_t>(t) * ntt31::PINV;
    const uint64_t u = t + static_cast<uint64_t>(m) * ntt31::P;
    return reduce_2p(static_cast<uint32_t>(u >> 32));
}

// Multiply by the compile-time twiddle W_M^E (forward: omega_M^E, inverse:
// omega_M^-E; omega_M = psi^(2048/M)), data in normal form.
template <int M, int E, bool INV>
__device__ __forceinline__ uint32_t ntt_twiddle_const(uint32_t v)
{
    constexpr int e = ((E % M) + M) % M;
    if constexpr (e == 0) {
        return v;
    }
    else if constexpr (2 * e == M) {
        return mod_sub(0u, v);
    }
    else {
        constexpr int64_t ex = static_cast<int64_t>(2048 / M) * e * (INV ? -1 : 1);
        constexpr uint32_t w = ntt31::to_mont_c(ntt31::psi_pow(ex));
        return mont_mul(v, w);
    }
}

// In-register M-point cyclic DFT mod P (radix-2 DIF, natural order), canonical
// inputs. A difference that a twiddle multiplies is not reduced first. LAZY: the
// outputs are below 2P, for a caller that multiplies them (a transform issues
// about 970 VALU instructions per lane for its butterflies and twiddles when
// every sum is reduced, 810 this way).
template <int M, bool INV, bool LAZY = false>
__device__ __forceinline__ void ntt_dft_reg(uint32_t* x)
{
    static_for<4>([&](auto sc) {
        constexpr int half = (M >> 1) >> decltype(sc)::value;
        if constexpr (half >= 1) {
#pragma unroll
            for (int start = 0; start < M; start += 2 * half) {
                static_for<half>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const uint32_t u = x[start + j];
                    const uint32_t v = x[start + j + half];
                    if constexpr (LAZY && half == 1)
                        x[start + j] = u + v;
                    else
                        x[start + j] = mod_add(u, v);
                    if constexpr (j != 0 || (LAZY && half == 1))
                        x[start + j + half] =
                            ntt_twiddle_const<M, j*(M / (2 * half)), INV>(u + ntt31::P - v);
                    else
                        x[start + j + half] = mod_sub(u, v);
                });
            }
        }
    });
    uint32_t tmp[M];
#pragma unroll
    for (int i = 0; i < M; i++) {
        int r = 0;
#pragma unroll
        for (int b = 1, s = M / 2; b < M; b <<= 1, s >>= 1)
            if (i & b) r |= s;
        tmp[r] = x[i];
    }
#pragma unroll
    for (int i = 0; i < M; i++) x[i] = tmp[i];
}

// Device tables (Montgomery form), built at init:
//   twl[k2*64 + l]  = psi^(l (1 + 2 k2))        forward step-2 twiddle x lane twist
//   twli[k2*64 + l] = psi^-(l (1 + 2 k2))       inverse
//   tw64[c*8 + a]   = omega^(16 a c)            (omega = psi^2; inverse: conjugate power)
//   tw64i[c*8 + a]  = omega^-(16 a c)
//   cr[r]  = psi^(64 r), cri[r] = psi^(-64 r) * N^-1   (r < 16)
//   pw[t]  = psi^t (t < 2048): evaluation-point powers for X^a - 1
struct NttTables {
    const uint32_t* twl;
    const uint32_t* twli;
    const uint32_t* tw64;
    const uint32_t* tw64i;
    const uint32_t* cr;
    const uint32_t* cri;
    const uint32_t* pw;
};

constexpr int kNttLdsWords = 16 * 72;  // per-wave scratch (transpose 1 needs 16 x 72)

// Scratch elements of the two transposes (4-byte elements, 64 banks; both
// sides of each are conflict-free). t1w/t1r: transpose 1 by register row k2 and
// by (group, step); t2a/t2c: transpose 2 with this lane's low digit as a or c.
struct NttPadded {
    uint32_t* lds;
    int lo, q, lane;
    __device__ __forceinline__ explicit NttPadded(uint32_t* p) : lds(p)
    {
        lane = threadIdx.x & 63;
        lo = lane & 7;
        q = lane >> 3;
    }
    __device__ __forceinline__ uint32_t& t1w(int k2) const { return lds[k2 * 72 + lane]; }
    __device__ __forceinline__ uint32_t& t1r(int g, int b) const
    {
        return lds[(g * 8 + q) * 72 + 8 * b + lo];
    }
    __device__ __forceinline__ uint32_t& t2(int g, int a, int c) const
    {
        return lds[(q * 2 + g) * 64 + 8 * ((a + q) & 7) + ((c + q) & 7)];
    }
    __device__ __forceinline__ uint32_t& t2a(int g, int c) const { return t2(g, lo, c); }
    __device__ __forceinline__ uint32_t& t2c(int g, int a) const { return t2(g, a, lo); }
};

// The same without padding: a wave's scratch is the size of its spectrum.
// Rows are swizzled by xor, so an element's address is one of four bases xor a
// constant; the bases are recomputed for each transform, because the addresses
// kept over a whole rotation (32 registers) spill at 128 registers a wave.
struct NttPacked {
    char* lds;  // LDS start that `base` counts from, in bytes
    uint32_t w1, r1, a2, c2;
    // base: a multiple of 4 KiB
    __device__ __forceinline__ NttPacked(void* p, uint32_t base) : lds(static_cast<char*>(p))
    {
        uint32_t lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const uint32_t lo = lane & 7, q = lane >> 3;
        w1 = base + lane * 4;
        r1 = w1 + q * 256;
        a2 = base + q * 512 + 32 * (lo ^ q) + 4 * q;
        c2 = base + q * 512 + 32 * q + 4 * (lo ^ q);
    }
    __device__ __forceinline__ uint32_t& at(uint32_t byte) const
    {
        return *reinterpret_cast<uint32_t*>(lds + byte);
    }
    __device__ __forceinline__ uint32_t& t1w(int k2) const
    {
        return at((w1 ^ (32 * (k2 & 7))) + 256 * k2);
    }
    __device__ __forceinline__ uint32_t& t1r(int g, int b) const
    {
        return at((r1 ^ (32 * b)) + 2048 * g);
    }
    __device__ __forceinline__ uint32_t& t2a(int g, int c) const { return at((a2 ^ (4 * c)) + 256 * g); }
    __device__ __forceinline__ uint32_t& t2c(int g, int a) const { return at((c2 ^ (32 * a)) + 256 * g); }
};

// Both transforms step their issue priority down (wave_prio), so that waves which
// meet at a barrier reach it together: rotations of 4096 jobs 8.82 -> 8.35 ms.
//
// Forward negacyclic NTT of x[r] = coefficient (lane + 64 r): x[0] in [0, P), the
// others any 32-bit value of their residue (they are multiplied first).
template <class Scratch>
__device__ __forceinline__ void ntt_forward(uint32_t (&x)[16], const Scratch& sc, const NttTables& tb)
{
    const int lane = threadIdx.x & 63;
    wave_prio<true>(3);
#pragma unroll
    for (int r = 1; r < 16; r++) x[r] = mont_mul(x[r], tb.cr[r]);
    ntt_dft_reg<16, false, true>(x);
#pragma unroll
    for (int k2 = 0; k2 < 16; k2++) x[k2] = mont_mul(x[k2], tb.twl[k2 * 64 + lane]);
#pragma unroll
    for (int k2 = 0; k2 < 16; k2++) sc.t1w(k2) = x[k2];
    wave_lds_sync();
    const int lo = lane & 7;
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int b = 0; b < 8; b++) x[g * 8 + b] = sc.t1r(g, b);
    wave_lds_sync();
    wave_prio<true>(2);
#pragma unroll
    for (int g = 0; g < 2; g++) {
        ntt_dft_reg<8, false, true>(&x[g * 8]);
        x[g * 8] = reduce_2p(x[g * 8]);
#pragma unroll
        for (int c = 1; c < 8; c++) x[g * 8 + c] = mont_mul(x[g * 8 + c], tb.tw64[c * 8 + lo]);
#pragma unroll
        for (int c = 0; c < 8; c++) sc.t2a(g, c) = x[g * 8 + c];
    }
    wave_lds_sync();
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int a = 0; a < 8; a++) x[g * 8 + a] = sc.t2c(g, a);
    wave_lds_sync();
    wave_prio<true>(1);
#pragma unroll
    for (int g = 0; g < 2; g++) ntt_dft_reg<8, false>(&x[g * 8]);
}

// Inverse (incl. N^-1): spectrum in the forward's register layout ->
// coefficients x[r] = coefficient (lane + 64 r), canonical.
template <class Scratch>
__device__ __forceinline__ void ntt_inverse(uint32_t (&x)[16], const Scratch& sc, const NttTables& tb)
{
    const int lane = threadIdx.x & 63;
    wave_prio<true>(3);
    const int lo = lane & 7;
#pragma unroll
    for (int g = 0; g < 2; g++) {
        ntt_dft_reg<8, true, true>(&x[g * 8]);
#pragma unroll
        for (int a = 0; a < 8; a++) sc.t2c(g, a) = x[g * 8 + a];
    }
    wave_lds_sync();
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int c = 0; c < 8; c++) x[g * 8 + c] = sc.t2a(g, c);
    wave_lds_sync();
    wave_prio<true>(2);
#pragma unroll
    for (int g = 0; g < 2; g++) {
        x[g * 8] = reduce_2p(x[g * 8]);
#pragma unroll
        for (int c = 1; c < 8; c++) x[g * 8 + c] = mont_mul(x[g * 8 + c], tb.tw64i[c * 8 + lo]);
        ntt_dft_reg<8, true, true>(&x[g * 8]);
#pragma unroll
        for (int b = 0; b < 8; b++) sc.t1r(g, b) = x[g * 8 + b];
    }
    wave_lds_sync();
#pragma unroll
    for (int k2 = 0; k2 < 16; k2++) x[k2] = sc.t1w(k2);
    wave_lds_sync();
    wave_prio<true>(1);
#pragma unroll
    for (int k2 = 0; k2 < 16; k2++) x[k2] = mont_mul(x[k2], tb.twli[k2 * 64 + lane]);
    ntt_dft_reg<16, true, true>(x);
#pragma unroll
    for (int r = 0; r < 16; r++) x[r] = mont_mul(x[r], tb.cri[r]);
}

__device__ __forceinline__ void ntt_forward(uint32_t (&x)[16], uint32_t* lds, const NttTables& tb)
{
    ntt_forward(x, NttPadded(lds), tb);
}
__device__ __forceinline__ void ntt_inverse(uint32_t (&x)[16], uint32_t* lds, const NttTables& tb)
{
    ntt_inverse(x, NttPadded(lds), tb);
}

// Reference conversions (include/ntt_small_modulus.cuh:284-361), lvl1 prime.
__device__ __forceinline__ uint32_t torus_to_ntt31(uint32_t a)
{
    // floor((a P + 2^31) / 2^32) in [0, P]; P itself is the residue 0
    const uint64_t v = (static_cast<uint64_t>(a) * ntt31::P + (1ULL << 31)) >> 32;
    return v >= ntt31::P ? static_cast<uint32_t>(v - ntt31::P) : static_cast<uint32_t>(v);
}
// v mod P for |v| < P: as u32 a negative v is above 2^31 > P and v + P
// wraps to P - |v|, so the unsigned min picks the residue either way
// (two VALU ops, no compare and select).
__device__ __forceinline__ uint32_t signed_to_ntt31(int32_t v)
{
    const uint32_t u = static_cast<uint32_t>(v);
    return __builtin_elementwise_min(u, u + ntt31::P);
}
__device__ __forceinline__ uint32_t ntt31_to_torus32(uint32_t val)
{
    // round(mag floor(2^63 / P) / 2^31): the factor is 2^32 + c with a small c,
    // and mag 2^32 / 2^31 is an integer
    constexpr uint32_t c = static_cast<uint32_t>((1ULL << 63) / ntt31::P - (1ULL << 32));
    const uint32_t minus = ntt31::P - val;
    const bool neg = val > ntt31::HALF_P;
    const uint32_t mag = neg ? minus : val;
    const uint64_t low = static_cast<uint64_t>(mag) * c + (1ULL << 30);
    const uint32_t t32 = 2u * mag + static_cast<uint32_t>(low >> 31);
    return neg ? 0u - t32 : t32;
}

}  // namespace cufhe_amd
