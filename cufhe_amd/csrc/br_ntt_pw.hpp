// NTT-backend blind rotation of up to eight jobs by one workgroup, the products
// split over the waves by bins (the batched form's NTT kernel).
//
// Arithmetic: the step of br_ntt.hpp (reference
// include/gatebootstrapping_gpu.cuh:522-797, :1187-1332; drivers :801-884) for
// the three modes -- plain CMUX, 2-bit key bundle, block-binary. Everything is
// an exact residue, so any grouping of the sums gives the same words.
//
// What bounds it: VALU issue of integer instructions (a 32 x 32 multiply-add
// issues at the rate of an addition, so the count of all of them matters; four
// waves per SIMD keep the unit busy, about 3900 instructions a wave and
// block-binary step). Two waves per job that each own an output column, as in
// br_ntt.hpp, derive every X^a - 1 root and read every key word for themselves
// and reduce every key sum. Here
//  - wave 2 s + j transforms the digits of component j of job s (two forward,
//    one inverse transform a step), but between the step's two barriers it owns
//    one register row of 64 bins of ALL jobs: a key word is loaded once per
//    workgroup, straight into a VGPR and one phase ahead, and a root is one table
//    read (psi^t - 1, no multiply) instead of a Montgomery product per digit and
//    column;
//  - the sum over rows is taken before the sum over keys,
//      s_col = sum_e (X^a_e - 1) * ( sum_{comp,q} D_{comp,q} K_e(comp, q, col) ),
//    so that four products share one reduction: for four keys 40 products and 10
//    reductions a bin and job instead of 56 products and 36;
//  - a transform swizzles its first transpose instead of padding it, so its
//    scratch is its spectrum's place; the two output columns of a bin replace
//    digit 0 of the same bin. Eight jobs and the tables are 155 KiB.
// All sixteen waves share the products also when fewer jobs rotate, which
// shortens a short batch's step.
//
// Measured against two waves per job and two jobs per workgroup (rotations of
// 1 / 1024 / 4096 jobs, ms): block-binary 2.92 / 4.28 / 14.1 -> 1.29 / 2.30 / 8.34,
// key bundle 5.19 / 7.79 / 25.8 -> 2.46 / 4.49 / 16.5, plain 9.14 / 12.3 / 38.4 ->
// 4.62 / 7.70 / 27.4.
#pragma once

#include "br_ntt.hpp"
#include "launch_rules.hpp"

namespace cufhe_amd {

template <int MODE>
struct NttModeShape {
    static constexpr int NK = MODE == NTT_PLAIN ? 1 : (MODE == NTT_KB ? 3 : kBlockEll);
    static constexpr int STEP_TRGSW = NK;
    static constexpr int STEP_BITS = MODE == NTT_PLAIN ? 1 : (MODE == NTT_KB ? 2 : kBlockEll);
    static constexpr int STEPS = lvl0param::n / STEP_BITS;
};

// two waves a job, sixteen rows of bins
constexpr int kNttPwThreads = 128 * kNttPwJobs;

struct NttPwShared {
    static constexpr int C = kNttPwJobs, n0 = lvl0param::n, L = lvl1param::l;
    // per wave (job s, component j: 2 s + j): its digit spectra; transform
    // scratch; digit 0 then holds output column j
    uint32_t spec[2 * C][L][lvl1param::n];
    uint32_t twl[16 * 64], twli[16 * 64], tw64[64], tw64i[64], cr[16], cri[16];
    int32_t root[2 * lvl1param::n];  // psi^t - 1, Montgomery form, in [-P/2, P/2]
    uint16_t abar[C][n0 + 4];        // mod-switched lvl0 mask
    uint32_t bar[C];
    uint32_t corr[C][2];  // block-binary correction partial sums (one per wave)
};

// t R^-1 mod P, canonical, for t <= 4 (P - 1)^2 (a sum of up to four products of
// residues: 4 P^2 < 2^64 and its upper word is below 2P). The low words of t and
// m P are equal, so only the upper words are subtracted.
__device__ __forceinline__ uint32_t ntt_dot_reduce(uint64_t t)
{
    const uint32_t m = static_cast<uint32_t>(t) * (0u - ntt31::PINV);
    const uint32_t h = __umulhi(m, ntt31::P);  // < P
    const uint32_t r = reduce_2p(static_cast<uint32_t>(t >> 32)) - h;
    return __builtin_elementwise_min(r, r + ntt31::P);
}

// The same residue, not canonical: in (-P, P).
__device__ __forceinline__ int32_t ntt_dot_signed(uint64_t t)
{
    const uint32_t m = static_cast<uint32_t>(t) * (0u - ntt31::PINV);
    return static_cast<int32_t>(reduce_2p(static_cast<uint32_t>(t >> 32)) - __umulhi(m, ntt31::P));
}
// t R^-1 mod P, canonical, for |t| < 2 P^2 (upper word within P of zero).
__device__ __forceinline__ uint32_t ntt_dot_reduce(int64_t t)
{
    const uint32_t m = static_cast<uint32_t>(t) * (0u - ntt31::PINV);
    const uint32_t hi = signed_to_ntt31(static_cast<int32_t>(t >> 32));
    const uint32_t r = hi - __umulhi(m, ntt31::P);
    return __builtin_elementwise_min(r, r + ntt31::P);
}

// Rotates the workgroup's `live` jobs. The waves of the other slots transform
// nothing, but take their row of the products.
template <int MODE>
__device__ __forceinline__ void blind_rotate_ntt_pw(NttPwShared& sm, int live, int slot, int j,
                                                    uint32_t mu, uint32_t (&acc)[16],
                                                    const NttKeys& K)
{
    using P = lvl1param;
    using S = NttModeShape<MODE>;
    constexpr int N = P::n, L = P::l, NK = S::NK;
    constexpr int NCOMP = 2;
    static_assert(2 * kNttPwJobs == 16, "one register row of bins a wave");
    static_assert(L * NCOMP <= 4 && NK <= 4, "sums of at most four products per reduction");
    const int lane = threadIdx.x & 63;
    const int wave = 2 * slot + j;
    uint32_t(*const my)[N] = sm.spec[wave];
    const uint32_t wave_base = wave * L * N * 4;
    const NttTables tb{sm.twl, sm.twli, sm.tw64, sm.tw64i, sm.cr, sm.cri, nullptr};

    const bool rotating = slot < live;
    const uint32_t bar = rotating ? sm.bar[slot] : 0u;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int i = ntt_coef_index(r, lane);
        if (j == 0)
            acc[r] = 0;
        else if (bar == 2 * N)
            acc[r] = mu;
        else
            acc[r] = ((static_cast<uint32_t>(i) < (bar & (N - 1))) ^ ((bar >> P::nbit) != 0)) ? 0u - mu
                                                                                          : mu;
    }

    // key words of this wave's row of bins: [key][component][digit][column]
    const int d = wave;
    const uint32_t* const key = K.bk + d * 64 + lane;
    // bin of register d of this lane (ntt_forward's output order)
    const uint32_t k2p1 = 2u * ((lane >> 3) + 8 * (d >> 3) + 16 * ((lane & 7) + 8 * (d & 7))) + 1u;
    uint32_t kv[NK][NCOMP][L][2];
    auto load_keys = [&](int it) {
        const uint32_t* p = key + static_cast<size_t>(it) * S::STEP_TRGSW * kTrgswNtt;
#pragma unroll
        for (int e = 0; e < NK; e++)
#pragma unroll
            for (int comp = 0; comp < NCOMP; comp++)
#pragma unroll
                for (int q = 0; q < L; q++)
#pragma unroll
                    for (int col = 0; col < 2; col++)
                        kv[e][comp][q][col] = p[e * kTrgswNtt + ((comp * L + q) * 2 + col) * N];
    };
    load_keys(0);

#pragma unroll 1
    for (int it = 0; it < S::STEPS; it++) {
        if (rotating) {
            // digit source: acc (KB, BB) or (X^a - 1) acc (plain)
            uint32_t src[16];
            if constexpr (MODE == NTT_PLAIN) {
                const uint32_t a0 = __builtin_amdgcn_readfirstlane(sm.abar[slot][it]);
#pragma unroll
                for (int r = 0; r < 16; r++) my[0][ntt_coef_index(r, lane)] = acc[r];
                wave_lds_sync();
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int i = ntt_coef_index(r, lane);
                    const uint32_t v = my[0][(i - static_cast<int>(a0)) & (N - 1)];
                    const bool neg =
                        (static_cast<uint32_t>(i) < (a0 & (N - 1))) ^ ((a0 >> P::nbit) != 0);
                    src[r] = (neg ? 0u - v : v) - acc[r];
                }
                wave_lds_sync();
            }
            else {
#pragma unroll
                for (int r = 0; r < 16; r++) src[r] = acc[r];
            }
#pragma unroll 1
            for (int q = 0; q < L; q++) {
                uint32_t x[16];
#pragma unroll
                for (int r = 1; r < 16; r++)
                    x[r] = static_cast<uint32_t>(Gadget<P>::digit(src[r], q)) + ntt31::P;
                x[0] = signed_to_ntt31(Gadget<P>::digit(src[0], q));
                ntt_forward(x, NttPacked(sm.spec, wave_base + q * N * 4), tb);
#pragma unroll
                for (int r = 0; r < 16; r++) my[q][r * 64 + lane] = x[r];
            }
        }
        __syncthreads();  // every digit spectrum written
#pragma unroll 1
        for (int s = 0; s < live; s++) {
            int32_t rt[NK];
            if constexpr (MODE != NTT_PLAIN) {
                uint32_t a[NK];
                if constexpr (MODE == NTT_KB) {
                    // key order of the bundle: both bits, first, second
                    a[1] = sm.abar[s][2 * it];
                    a[2] = sm.abar[s][2 * it + 1];
                    a[0] = a[1] + a[2];
                }
                else {
#pragma unroll
                    for (int e = 0; e < NK; e++) a[e] = sm.abar[s][it * NK + e];
                }
#pragma unroll
                for (int e = 0; e < NK; e++)
                    rt[e] = sm.root[__umul24(a[e], k2p1) & (2 * N - 1)];
            }
            uint32_t D[NCOMP][L];
#pragma unroll
            for (int comp = 0; comp < NCOMP; comp++)
#pragma unroll
                for (int q = 0; q < L; q++) D[comp][q] = sm.spec[2 * s + comp][q][d * 64 + lane];
#pragma unroll
            for (int col = 0; col < 2; col++) {
                int64_t sum = 0;
                uint32_t r = 0;
#pragma unroll
                for (int e = 0; e < NK; e++) {
                    uint64_t t = 0;
#pragma unroll
                    for (int comp = 0; comp < NCOMP; comp++)
#pragma unroll
                        for (int q = 0; q < L; q++)
                            t += static_cast<uint64_t>(D[comp][q]) * kv[e][comp][q][col];
                    if constexpr (MODE == NTT_PLAIN)
                        r = ntt_dot_reduce(t);
                    else
                        sum += static_cast<int64_t>(rt[e]) * ntt_dot_signed(t);
                }
                if constexpr (MODE != NTT_PLAIN) r = ntt_dot_reduce(sum);
                if constexpr (MODE == NTT_KB) {
                    // the bundle's gadget identity term
                    uint64_t t = 0;
#pragma unroll
                    for (int q = 0; q < L; q++)
                        t += static_cast<uint64_t>(D[col][q]) * K.one_mont[q];
                    r = mod_add(r, ntt_dot_reduce(t));
                }
                sm.spec[2 * s + col][0][d * 64 + lane] = r;
            }
        }
        load_keys(it + 1 < S::STEPS ? it + 1 : it);  // the last step reloads its own
        __syncthreads();  // every output column written
        if (rotating) {
            uint32_t s[16];
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = my[0][r * 64 + lane];
            wave_lds_sync();
            ntt_inverse(s, NttPacked(sm.spec, wave_base), tb);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t t = ntt31_to_torus32(s[r]);
                acc[r] = MODE == NTT_KB ? t : acc[r] + t;
            }
        }
    }
}

}  // namespace cufhe_amd
