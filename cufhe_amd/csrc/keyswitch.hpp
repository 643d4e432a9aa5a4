// Identity key switching lvl1 -> lvl0 and lvl2 -> lvl0 with the gate's
// linear combination fused in front.
//
// Reference: include/keyswitch_gpu.cuh:13-23 (iksoffsetgen), :33-50
// (KeySwitchTorusConvert), :128-187 (KeySwitchFromTLWE), :189-256
// (IdentityKeySwitchPreAdd). For each output coefficient i in [0, n0]:
//   res = (i == n0) ? conv(ca*in0[dn] + cb*in1[dn] + offset)
//                   : (subset && i < n0 ? conv(ca*in0[i] + cb*in1[i]) : 0)
//   for each switched input coefficient j (all, or j >= n0 when subset):
//     tmp = ca*in0[j] + cb*in1[j] + decomp_offset + round_offset
//     for each of t signed digits v of basebit bits (most significant first):
//       res -= sign(v) * KSK[j'][digit][|v|-1][i]      (j' = j - first)
// KSK layout: [switched j][t][2^(basebit-1)][n0+1] uint32.
#pragma once

#include "device_common.hpp"

namespace cufhe_amd {

template <class KS>
struct KsTraits {
    using DT = typename KS::domainP::T;
    static constexpr int W = kTorusBits<DT>;
    static constexpr uint32_t dn = KS::domainP::k * KS::domainP::n;
    static constexpr uint32_t n0 = KS::targetP::k * KS::targetP::n;
    static constexpr uint32_t numbase = 1u << (KS::basebit - 1);
    static constexpr DT decomp_offset()
    {
        DT o = 0;
        for (uint32_t i = 1; i <= KS::t; i++)
            o += static_cast<DT>(numbase) << (W - i * KS::basebit);
        return o;
    }
    static constexpr DT kRound =
        (KS::basebit * KS::t) < static_cast<uint32_t>(W)
            ? static_cast<DT>(1) << (W - (1 + KS::basebit * KS::t))
            : 0;
    static constexpr DT kOffset = decomp_offset() + kRound;
    __device__ __forceinline__ static uint32_t convert(DT v)
    {
        if constexpr (W == 32)
            return static_cast<uint32_t>(v);
        else
            return static_cast<uint32_t>((v + (static_cast<DT>(1) << 31)) >> 32);
    }
    static constexpr size_t row_words = n0 + 1;
    static constexpr size_t digit_words = numbase * row_words;
    static constexpr size_t coef_words = KS::t * digit_words;
};

// Key switch of the combination ca*in0 + cb*in1 (+offset on the body) for
// one job, spread over NW waves of a workgroup: wave w takes the switched
// coefficients j in its 1/NW share, each lane accumulates output columns
// lane + 64 c (c < 10), the partial sums go through red[NW][n0 + 1] in LDS,
// and threads [0, 64 NW) sum them into out. Integer sums mod 2^32, so the
// split does not change a bit.
// A job reads dn x t KSK rows of 2.5 KB (18 MB at lvl1), so one CU is bound by
// its L2 -> VGPR path, and before that by latency: the t rows of a coefficient
// are loaded together, one coefficient ahead of their sums, and the digits of
// 64 coefficients are prepared by the lanes and read back one by one. With each
// row's loads next to its sums one lvl1 job took 459 us, 1024 took 627 and 4096
// 4420; now 144, 538 and 2138 (1024 jobs: 24 TB/s out of the L2s).
// `wave` is the wave's index within the NW waves of this job; every thread
// of the workgroup must call it (one __syncthreads inside).
template <class KS, bool SUBSET, int NW>
__device__ __forceinline__ void key_switch_waves(uint32_t* out, const typename KS::domainP::T* in0,
                                                 const typename KS::domainP::T* in1, int32_t ca,
                                                 int32_t cb, typename KS::domainP::T offset,
                                                 const uint32_t* ksk, uint32_t* red, int wave,
                                                 int lane)
{
    using TR = KsTraits<KS>;
    using DT = typename TR::DT;
    constexpr uint32_t first = SUBSET ? TR::n0 : 0;
    constexpr int NC = (TR::n0 + 1 + 63) / 64;
    constexpr uint32_t share = (TR::dn - first + NW - 1) / NW;
    const DT ua = static_cast<DT>(static_cast<std::make_signed_t<DT>>(ca));
    const DT ub = static_cast<DT>(static_cast<std::make_signed_t<DT>>(cb));
    uint32_t res[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int i = lane + 64 * c;
        uint32_t r = 0;
        if (wave == 0) {  // base terms once
            if (i == static_cast<int>(TR::n0)) {
                DT v = ua * in0[TR::dn] + offset;
                if (in1) v += ub * in1[TR::dn];
                r = TR::convert(v);
            }
            else if (SUBSET && i < static_cast<int>(TR::n0)) {
                DT v = ua * in0[i];
                if (in1) v += ub * in1[i];
                r = TR::convert(v);
            }
        }
        res[c] = r;
    }
    const uint32_t j0 = first + static_cast<uint32_t>(wave) * share;
    const uint32_t j1 = j0 + share < TR::dn ? j0 + share : TR::dn;
    constexpr uint32_t kDigits = KS::t * KS::basebit;  // bits of all digits of a coefficient
    static_assert(KS::basebit == 2 && kDigits <= 32, "digits in {-2, .., 1}, packed in a word");
    struct Rows {
        uint32_t x[KS::t][NC];
    };
    // the rows of a coefficient's nonzero digits
    auto load = [&](uint32_t j, uint32_t digits) {
        const uint32_t* kj = ksk + static_cast<size_t>(j - first) * TR::coef_words;
        Rows r;
#pragma unroll
        for (uint32_t k = 0; k < KS::t; k++) {
            const uint32_t v = (digits >> (kDigits - (k + 1) * KS::basebit)) & 3u;
            if (v != 2) {
                const uint32_t* row = kj + k * TR::digit_words + (v == 0 ? TR::row_words : 0);
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    const int i = lane + 64 * c;
                    r.x[k][c] = row[i <= static_cast<int>(TR::n0) ? i : static_cast<int>(TR::n0)];
                }
            }
        }
        return r;
    };
    auto add = [&](const Rows& r, uint32_t digits) {
#pragma unroll
        for (uint32_t k = 0; k < KS::t; k++) {
            const uint32_t v = (digits >> (kDigits - (k + 1) * KS::basebit)) & 3u;
            if (v < 2) {  // digit -2 or -1
#pragma unroll
                for (int c = 0; c < NC; c++) res[c] += r.x[k][c];
            }
            else if (v == 3) {  // digit 1
#pragma unroll
                for (int c = 0; c < NC; c++) res[c] -= r.x[k][c];
            }
        }
    };
    for (uint32_t base = j0; base < j1; base += 64) {
        uint32_t mine = 0;
        const uint32_t jl = base + static_cast<uint32_t>(lane);
        if (jl < j1) {
            DT tmp = ua * in0[jl] + TR::kOffset;
            if (in1) tmp += ub * in1[jl];
            mine = static_cast<uint32_t>(tmp >> (TR::W - kDigits)) & ((1u << kDigits) - 1);
        }
        const uint32_t n = j1 - base < 64 ? j1 - base : 64;
        // digits of coefficient base + i (wave-uniform); the last one again past the end
        auto at = [&](uint32_t i) {
            return static_cast<uint32_t>(__builtin_amdgcn_readlane(mine, i < n ? i : n - 1));
        };
        auto index = [&](uint32_t i) { return base + (i < n ? i : n - 1); };
        uint32_t da = at(0), db;
        Rows a = load(index(0), da), b;
#pragma unroll 1
        for (uint32_t i = 0; i < n; i += 2) {
            db = at(i + 1);
            b = load(index(i + 1), db);
            asm volatile("" ::: "memory");  // the loads stay ahead of the sums
            add(a, da);
            da = at(i + 2);
            a = load(index(i + 2), da);
            asm volatile("" ::: "memory");
            if (i + 1 < n) add(b, db);
        }
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int i = lane + 64 * c;
        if (i <= static_cast<int>(TR::n0)) red[wave * (TR::n0 + 1) + i] = res[c];
    }
    __syncthreads();
    const int tid = wave * 64 + lane;
    for (int i = tid; i <= static_cast<int>(TR::n0); i += 64 * NW) {
        uint32_t r = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) r += red[w * (TR::n0 + 1) + i];
        out[i] = r;
    }
}

}  // namespace cufhe_amd
