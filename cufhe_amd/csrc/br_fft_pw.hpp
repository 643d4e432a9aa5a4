// Key-bundle blind rotation with the digit transforms of a job spread over
// several waves and the multiply-accumulate split over all waves by spectrum
// bins.
//
// Arithmetic: br_fft.hpp's key-bundle step (reference
// include/gatebootstrapping_gpu.cuh:895-1033 AccumulateKeyBundle and
// :1335-1429 the drivers). At lvl2 operation for operation, so the outputs are
// bit-identical to k_br_fft. At lvl1 the external product is an integer that
// FP64 leaves within a small fraction of a unit, so any order of operations
// rounds to the same words: there the transforms are fft512.hpp's and
// X^(a0+a1) is the product of X^a0 and X^a1.
//
// A step has three phases, each ended by a workgroup barrier:
//  1. forward: wave (job, component j, qi) turns its DPW digit polynomials
//     into spectra, each in an LDS buffer that is the transform's scratch too;
//  2. multiply-accumulate: every wave takes R/W registers' worth of bins
//     (64 bins each) of its jobs. A key value is loaded from L2 by one wave,
//     straight into VGPRs, and used for every job: there is no key ring in LDS
//     and no barrier inside the phase. A lane reads the digit spectra at its
//     bins and writes the two output spectra over two of them (no other lane
//     touches those bins);
//  3. inverse: wave qi = 0 of (job, j) transforms component j's output back,
//     rounds, and hands the next digits to its partner waves through their idle
//     buffers; a partner (or the wave itself) prepares the next step's roots.
// What bounds it: FP64 issue and LDS traffic, about equally, over the whole
// CU. (An LDS KiB costs a CU 5.7 ns written and 3.2 ns read, a wave's FP64
// instruction 0.5 ns; FP64 MFMA runs on the same pipe as the vector FMAs.)
#pragma once

#include "br_fft.hpp"
#include "fft512.hpp"

namespace cufhe_amd {

// J jobs per workgroup; DPW digit polynomials per wave and pass; the L gadget
// digits go through phases 1-2 in PASSES passes (fewer digit buffers in LDS,
// the sums stay in VGPRs between them); PF key blocks (three values) are in
// flight per lane.
template <class P_, int J_, int PASSES_, int DPW_, int PF_, int HELP_ = 0>
struct PwShape {
    using P = P_;
    using T = typename P::T;
    static constexpr int N = P::n, H = N / 2, R = H / 64, G = R / 8, L = P::l;
    static constexpr bool kLvl1 = sizeof(T) == 4;
    static constexpr int J = J_, PASSES = PASSES_, DPW = DPW_, PF = PF_;
    static constexpr int QD = L / PASSES;  // digits per component and pass
    static constexpr int QW = QD / DPW;    // digit waves per component
    static constexpr int WPJ = 2 * QW, FW = J * WPJ;  // transform waves
    static constexpr int HELP = HELP_;                // waves of phase 2 only, and the roots
    static constexpr int W = FW + HELP, NT = 64 * W;
    static constexpr int SETS = W > R ? W / R : 1;  // wave sets that share the bins
    static constexpr int JL = J / SETS;             // jobs per wave in phase 2
    static constexpr int BPL = W > R ? 1 : R / W;   // registers (64-bin groups) per wave
    static constexpr int BLK = QD * 4;              // key blocks per pass and register
    static constexpr int NB = BPL * BLK;            // key blocks per pass
    static constexpr int STEPS = lvl0param::n / 2;
    // root sets in LDS: lvl1 forms X^(a0+a1) as a product, lvl2 reads it from the table
    static constexpr int NX = kLvl1 ? 2 : 3;
    // digit words per lane: lvl1 packs both digits of two coefficients
    static constexpr int WORDS = kLvl1 ? R : R * PASSES;
    static constexpr bool kPrio = J > 1;  // several waves per SIMD meet at the barriers
    // all key blocks of a step in flight before phase 2 (else PF ahead, rolling)
    static constexpr bool kFull = PASSES == 1 && PF == NB;
    // the roots of a job in the idle ends of its digit 1 buffers instead of an array
    static constexpr bool kTail = kLvl1 && QW == 2 && HELP == 0;
    static constexpr int TAB = kLvl1 ? fft512::kTabWords : 3 * 64;
    static_assert(QW * DPW == QD && QD * PASSES == L && JL * SETS == J, "shape");
    static_assert(kLvl1 || DPW == 1, "lvl2 packs one digit per word half");
    static_assert(HELP == 0 || HELP >= 2 * J, "two root waves per job");
    static_assert(!kFull || kLvl1, "the next step's keys are loaded in fft512's hooks");
    static_assert((W > R ? W % R == 0 : R % W == 0) && NB % PF == 0, "even split");
};

template <class S>
struct PwShared {
    cplx buf[S::J * 2 * S::QD][fft_stage::kScratchPad(S::H)];  // [(job * QD + digit) * 2 + j]
    cplx base[S::kTail ? 1 : S::J][S::NX][S::G][S::kTail ? 1 : 64];                          // E[a (1 - 4 kb)] of a0, a1 (, a0 + a1)
    cplx tab[S::TAB];                                          // transform tables
    uint32_t a[S::J][S::NX];
};

template <class S>
struct PwWave {
    using P = typename S::P;
    using T = typename S::T;
    static constexpr int N = S::N, H = S::H, R = S::R, L = S::L;
    PwShared<S>& sm;
    const FourierKeys<P>& K;
    const int wave, lane;
    // transform wave: its job, component and digit wave; helpers: qi = -1 and
    // the job and component whose roots they prepare
    const int slot, j, qi;
    const bool rooter;  // prepares roots
    uint32_t words[S::WORDS];  // this wave's digits

    // Inverse waves (qi = 0) of odd and even jobs sit on different SIMDs.
    __device__ __forceinline__ PwWave(PwShared<S>& s, const FourierKeys<P>& k, int w, int ln)
        : sm(s), K(k), wave(w), lane(ln), slot(w < S::FW ? w / S::WPJ : ((w - S::FW) >> 1) % S::J), j(w & 1),
          qi(w >= S::FW ? -1 : ((w % S::WPJ) >> 1) ^ (S::QW == 2 ? (slot & 1) : 0)),
          rooter(S::HELP ? w >= S::FW && w < S::FW + 2 * S::J : qi == (S::QW == 1 ? 0 : 1))
    {
    }
    __device__ __forceinline__ cplx* buf(int s, int comp, int ql) const
    {
        return sm.buf[(s * S::QD + ql) * 2 + comp];
    }
    // Tables behind an offset the compiler cannot see through: their loads
    // stay inside the loop instead of occupying VGPRs across it.
    __device__ __forceinline__ const cplx* tables() const
    {
        int zo = 0;
        asm volatile("" : "+s"(zo));
        return sm.tab + zo;
    }
    __device__ __forceinline__ FFTTables lvl2_tables() const
    {
        const cplx* t = tables();
        return FFTTables{t, t + 64, nullptr, t + 128};
    }
    // cr[r] by scalar loads: wave-uniform operands that take no VGPRs
    __device__ __forceinline__ cplx cr(int r) const
    {
        using cptr = const __attribute__((address_space(4))) double*;
        const cptr p = (cptr)(reinterpret_cast<uintptr_t>(K.fft.cr));
        return cplx{p[2 * r], p[2 * r + 1]};
    }
    __device__ __forceinline__ void load_tables(int t)
    {
        if constexpr (S::kLvl1) {
            for (int i = t; i < fft512::kTabWords; i += S::NT) sm.tab[i] = K.fft.roots[i];
        }
        else {
            for (int i = t; i < 64; i += S::NT) {
                sm.tab[i] = K.fft.twl[i];
                sm.tab[64 + i] = K.fft.tw64[i];
                sm.tab[128 + i] = K.fft.tws[i];
            }
        }
    }

    // The words of digit wave q_ for coefficients lo (r) and hi (R + r).
    __device__ __forceinline__ static uint32_t pack(T lo, T hi, int q_, int pass)
    {
        if constexpr (S::kLvl1) {
            // bytes 3 and 2 of c + offset are the digits + 128
            const uint32_t a = lo + Gadget<P>::kOffset, b = hi + Gadget<P>::kOffset;
            return ((a >> 16) | (b & 0xffff0000u)) ^ 0x80808080u;
        }
        else {
            const int q = pass * S::QD + q_;
            return (static_cast<uint32_t>(Gadget<P>::digit(lo, q)) & 0xffffu) |
                   (static_cast<uint32_t>(Gadget<P>::digit(hi, q)) << 16);
        }
    }
    // folded digit m of this wave (lvl1: gadget digit qi * DPW + m) at register r
    __device__ __forceinline__ cplx digits(int r, int pass, int m) const
    {
        if constexpr (S::kLvl1) {
            const uint32_t sh = 8 * (1 - (qi * S::DPW + m));
            return cplx{static_cast<double>(static_cast<int32_t>(__builtin_amdgcn_sbfe(words[r], sh, 8))),
                        static_cast<double>(
                            static_cast<int32_t>(__builtin_amdgcn_sbfe(words[r], sh + 16, 8)))};
        }
        else {
            uint32_t u = words[r];
#pragma unroll
            for (int p = 1; p < S::PASSES; p++)
                if (p == pass) u = words[p * R + r];
            const int32_t w = static_cast<int32_t>(u);
            return cplx{static_cast<double>(static_cast<int16_t>(w)), static_cast<double>(w >> 16)};
        }
    }
    __device__ __forceinline__ void init_digits(uint32_t bar, T mu)
    {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i0 = lane + 64 * r;
            const T lo = j == 0 ? T(0) : test_vector_coef<P>(i0, bar, mu);
            const T hi = j == 0 ? T(0) : test_vector_coef<P>(i0 + H, bar, mu);
#pragma unroll
            for (int p = 0; p < S::WORDS / R; p++) words[p * R + r] = pack(lo, hi, qi, p);
        }
    }

    // Roots of this job's next step, gathered by the two waves (j = 0, 1) with
    // qi = RW: j = 0 takes a0 (and a0 + a1), j = 1 takes a1.
    struct Gathered {
        cplx v[2][S::G];
        uint32_t a0, a1;
    };
    __device__ __forceinline__ Gathered gather(uint32_t a0, uint32_t a1) const
    {
        Gathered r;
        r.a0 = a0;
        r.a1 = a1;
        const int c = lane & 7, q = lane >> 3;
#pragma unroll
        for (int g = 0; g < S::G; g++) {
            const int kb = (q + 8 * g) + R * c;
            const int t = static_cast<int>(j == 0 ? a0 : a1) * (1 - 4 * kb);
            r.v[0][g] = K.e2n[t & (2 * N - 1)];
            if constexpr (S::NX == 3)
                if (j == 0) r.v[1][g] = K.e2n[static_cast<int>(a0 + a1) * (1 - 4 * kb) & (2 * N - 1)];
        }
        return r;
    }
    __device__ __forceinline__ const cplx* root(int job, int m, int g) const
    {
        if constexpr (S::kTail)
            return buf(job, m, 1) + H;
        else
            return sm.base[job][m][g];
    }
    __device__ __forceinline__ void put(const Gathered& r)
    {
        if constexpr (S::kTail) {
            // the roots themselves follow behind the forward transform
            if (lane == 0) sm.a[slot][j] = j == 0 ? r.a0 : r.a1;
            return;
        }
#pragma unroll
        for (int g = 0; g < S::G; g++) {
            lds_store(&sm.base[slot][j][g][lane], r.v[0][g]);
            if constexpr (S::NX == 3)
                if (j == 0) lds_store(&sm.base[slot][2][g][lane], r.v[1][g]);
        }
        if (lane == 0) {
            sm.a[slot][j] = j == 0 ? r.a0 : r.a1;
            if constexpr (S::NX == 3)
                if (j == 0) sm.a[slot][2] = r.a0 + r.a1;
        }
    }

    // Key block b of a pass: register dd, digit, component, output column; its
    // three bundle members.
    struct KeyBlk {
        cplx k[3];
    };
    __device__ __forceinline__ KeyBlk load_key(int step, int pass, int b, int d0) const
    {
        constexpr size_t TS = kTrgswFourier<P>;
        const int dd = b / S::BLK, ql = (b % S::BLK) / 4, comp = (b / 2) & 1, col = b & 1;
        // wave-uniform address (SGPRs) plus the lane's 32-bit byte offset
        const uint32_t st = __builtin_amdgcn_readfirstlane(step);
        const uint32_t in_step = __builtin_amdgcn_readfirstlane(
            ((comp * L + pass * S::QD + ql) * 2 + col) * H + (d0 + dd) * 64);
        const uint64_t u = reinterpret_cast<uint64_t>(K.bk + st * (3 * TS) + in_step);
        using gbytes = const __attribute__((address_space(1))) char*;
        const gbytes p = (gbytes)(
            (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(u >> 32))) << 32) |
            static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(u))));
        const uint32_t off = static_cast<uint32_t>(lane) * sizeof(cplx);
        auto at = [&](size_t e) {
            typedef double v2 __attribute__((ext_vector_type(2)));
            const v2 v = *(const __attribute__((address_space(1))) v2*)(p + e * TS * sizeof(cplx) + off);
            return cplx{v.x, v.y};
        };
        return KeyBlk{{at(0), at(1), at(2)}};
    }

    // The rotation of the workgroup's jobs. abar(i): this wave's job's
    // mod-switched mask coefficient i (wave-uniform). live: whether this
    // wave's job exists. At the end the buffer of (job, j, digit 0) holds the N
    // coefficients of component j (visible to the wave with qi = 0).
    template <class Abar>
    __device__ __forceinline__ void rotate(bool live, uint32_t bar, T mu, Abar&& abar)
    {
        constexpr int PF = S::PF, NB = S::NB;
        const int set = S::W > R ? wave / R : 0;
        const int d0 = S::W > R ? wave % R : wave * S::BPL;
        const bool fft = live && qi >= 0;
        cplx* const mine = buf(slot, j, (qi < 0 ? 0 : qi) * S::DPW);
        const fft512::Slots slots = fft512::Slots::of(lane);
        uint32_t na0 = 0, na1 = 0;
        if (fft) init_digits(bar, mu);
        Gathered roots;
        if (live && rooter) {
            roots = gather(abar(0), abar(1));
            put(roots);
            na0 = abar(2);
            na1 = abar(3);
        }
        auto next_mask = [&](int it) {
            if (it + 2 < S::STEPS) {
                na0 = abar(2 * it + 4);
                na1 = abar(2 * it + 5);
            }
        };
        KeyBlk kv[PF];
        // full prefetch: transform waves that run the inverse load during the
        // next forward transform, the others during the inverse phase
        const bool early = !S::kFull || qi != 0;
        if (early) {
#pragma unroll
            for (int b = 0; b < PF; b++) kv[b] = load_key(0, 0, b, d0);
        }
        __syncthreads();  // the first roots
#pragma unroll 1
        for (int it = 0; it < S::STEPS; it++) {
            // the last blocks of a step prefetch the next step's first ones
            const int next = it + 1 < S::STEPS ? it + 1 : it;
            // W_8^(a d) of this step (scalar loads, long before their use)
            cplx w8[S::BPL][S::JL][S::NX];
#pragma unroll
            for (int jl = 0; jl < S::JL; jl++)
#pragma unroll
                for (int m = 0; m < S::NX; m++) {
                    const uint32_t a = __builtin_amdgcn_readfirstlane(sm.a[set * S::JL + jl][m]);
#pragma unroll
                    for (int dd = 0; dd < S::BPL; dd++) {
                        const int e = (a * static_cast<uint32_t>(d0 + dd)) & 7u;
                        w8[dd][jl][m] = cplx{kW8[e][0], kW8[e][1]};
                    }
                }
            const bool more = it + 1 < S::STEPS;
            if (S::HELP && live && rooter && more) {
                // helpers gather the next step's roots while the others transform
                roots = gather(na0, na1);
                next_mask(it);
            }
            cplx s[S::BPL][S::JL][2];
#pragma unroll
            for (int dd = 0; dd < S::BPL; dd++)
#pragma unroll
                for (int jl = 0; jl < S::JL; jl++) s[dd][jl][0] = s[dd][jl][1] = cplx{0.0, 0.0};
#pragma unroll 1
            for (int pass = 0; pass < S::PASSES; pass++) {
                const bool last = pass + 1 == S::PASSES;
                const int after = last ? next : it;
                const int after_pass = last ? 0 : pass + 1;
                if (fft) {
                    if constexpr (S::kLvl1) {
                        cplx z[S::DPW][8];
                        cplx* zb[S::DPW];
#pragma unroll
                        for (int m = 0; m < S::DPW; m++) {
                            zb[m] = buf(slot, j, qi * S::DPW + m);
#pragma unroll
                            for (int r = 0; r < 8; r++) z[m][r] = digits(r, pass, m);
                        }
                        // a third of the key blocks behind each stage's stores: the
                        // vector memory queue takes 16 cycles a load and CU
                        fft512::forward<S::DPW, S::kPrio>(z, zb, tables(), slots, lane, [&](int part) {
                            if constexpr (S::kFull)
                                if (qi == 0 || S::QW == 1)
#pragma unroll
                                    for (int b = 0; b < PF; b++)
                                        if (b * 3 / PF == part) kv[b] = load_key(it, 0, b, d0);
                        });
                    }
                    else {
                        using namespace fft_stage;
                        cplx z[R];
#pragma unroll
                        for (int r = 0; r < R; r++) z[r] = digits(r, pass, 0);
                        const FFTTables tb = lvl2_tables();
                        wave_prio<true>(3);
#pragma unroll
                        for (int r = 1; r < R; r++) z[r] = cmul(z[r], cr(r));
                        fwd_a_dft<R>(z, tb, lane);
                        t1_store<R, 2>(z, mine, lane);
                        wave_lds_sync();
                        t1_load<R, 2>(z, mine, lane);
                        wave_lds_sync();
                        wave_prio<true>(2);
                        fwd_b<R>(z, tb, lane);
                        t2_store_cx<R, 2>(z, mine, lane);
                        wave_lds_sync();
                        t2_load_xc<R, 2>(z, mine, lane);
                        wave_lds_sync();
                        wave_prio<true>(1);
                        fwd_c<R>(z);
                        wave_prio<true>(0);
#pragma unroll
                        for (int d = 0; d < R; d++) lds_store(&mine[d * 64 + lane], z[d]);
                    }
                }
                if constexpr (S::kTail)
                    if (live && rooter) lds_store(&mine[H + lane], roots.v[0][0]);
                if (!fft && S::kFull && !early) {
                    // no job: the wave still multiplies for the others
#pragma unroll
                    for (int b = 0; b < PF; b++) kv[b] = load_key(it, 0, b, d0);
                }
                // X^a - 1 at this wave's bins; the roots were published a barrier ago
                cplx x[S::BPL][S::JL][3];
                auto make_x = [&]() {
#pragma unroll
                for (int dd = 0; dd < S::BPL; dd++)
#pragma unroll
                    for (int jl = 0; jl < S::JL; jl++) {
                        cplx(&xx)[3] = x[dd][jl];
#pragma unroll
                        for (int m = 0; m < S::NX; m++)
                            xx[m] = cmul(lds_load(&root(set * S::JL + jl, m, (d0 + dd) >> 3)[lane]),
                                         w8[dd][jl][m]);
                        if constexpr (S::NX == 2) xx[2] = cmul(xx[0], xx[1]);
#pragma unroll
                        for (int m = 0; m < 3; m++) xx[m].x -= 1.0;
                    }
                };
                if constexpr (!S::kTail) make_x();
                __syncthreads();  // digit spectra are in LDS
                if constexpr (S::kTail) make_x();
                // the spectra of a (digit, component) are loaded while the one
                // before it is multiplied
                constexpr int DN = S::BPL * S::QD * 2;
                cplx D[2][S::JL];
                auto load_d = [&](int n, cplx(&dst)[S::JL]) {
                    const int dd = n / (2 * S::QD), ql = (n / 2) % S::QD, comp = n & 1;
#pragma unroll
                    for (int jl = 0; jl < S::JL; jl++)
                        dst[jl] = lds_load(&buf(set * S::JL + jl, comp, ql)[(d0 + dd) * 64 + lane]);
                };
                load_d(0, D[0]);
                wave_prio<S::kPrio>(3);
#pragma unroll
                for (int dd = 0; dd < S::BPL; dd++) {
#pragma unroll
                    for (int ql = 0; ql < S::QD; ql++) {
                        const double hq = ldexp(1.0, -static_cast<int>((pass * S::QD + ql + 1) * P::Bgbit));
#pragma unroll
                        for (int comp = 0; comp < 2; comp++) {
                            const int n = (dd * S::QD + ql) * 2 + comp;
                            if (n + 1 < DN) load_d(n + 1, D[(n + 1) & 1]);
                            if (n == DN / 4) wave_prio<S::kPrio>(2);
                            if (n == DN / 2) wave_prio<S::kPrio>(1);
                            if (n == DN * 3 / 4) wave_prio<S::kPrio>(0);
#pragma unroll
                            for (int col = 0; col < 2; col++) {
                                const int i = dd * S::BLK + ql * 4 + comp * 2 + col;
                                const KeyBlk cur = kv[i % PF];
                                if constexpr (!S::kFull)
                                    kv[i % PF] = i + PF < NB ? load_key(it, pass, i + PF, d0)
                                                             : load_key(after, after_pass, i + PF - NB, d0);
#pragma unroll
                                for (int jl = 0; jl < S::JL; jl++) {
                                    cplx k = {comp == col ? hq : 0.0, 0.0};
                                    cmac(k, cur.k[2], x[dd][jl][1]);
                                    cmac(k, cur.k[1], x[dd][jl][0]);
                                    cmac(k, cur.k[0], x[dd][jl][2]);
                                    cmac(s[dd][jl][col], D[n & 1][jl], k);
                                }
                                // the loads of later blocks stay behind this block's products
                                __builtin_amdgcn_sched_barrier(0);
                            }
                        }
                    }
                }
                if (!last) __syncthreads();  // spectra consumed
            }
#pragma unroll
            for (int dd = 0; dd < S::BPL; dd++)
#pragma unroll
                for (int jl = 0; jl < S::JL; jl++)
#pragma unroll
                    for (int col = 0; col < 2; col++)
                        lds_store(&buf(set * S::JL + jl, col, 0)[(d0 + dd) * 64 + lane], s[dd][jl][col]);
            __syncthreads();  // output spectra are in the digit 0 buffers
            if (S::HELP == 0 && live && rooter && more) {
                roots = gather(na0, na1);
                next_mask(it);
            }
            // (behind the roots' loads: they return in order)
            if (S::kFull && early) {
#pragma unroll
                for (int b = 0; b < PF; b++) kv[b] = load_key(next, 0, b, d0);
            }
            if (live && qi == 0) {
                cplx z[R];
                if constexpr (S::kLvl1) {
                    fft512::inverse<S::kPrio>(z, mine, tables(), slots, lane);
                }
                else {
                    using namespace fft_stage;
#pragma unroll
                    for (int d = 0; d < R; d++) z[d] = lds_load(&mine[d * 64 + lane]);
                    wave_lds_sync();
                    const FFTTables tb = lvl2_tables();
                    inv_a<R>(z);
                    t2_store_xc<R, 2>(z, mine, lane);
                    wave_lds_sync();
                    t2_load_cx<R, 2>(z, mine, lane);
                    wave_lds_sync();
                    inv_b<R>(z, tb, lane);
                    t1_store_inv<R, 2>(z, mine, lane);
                    wave_lds_sync();
                    t1_load_inv<R, 2>(z, mine, lane);
                    wave_lds_sync();
                    inv_c_dft<R>(z, tb, lane);
#pragma unroll
                    for (int r = 1; r < R; r++) z[r] = cmulc(z[r], cr(r));
                }
                // torus word of a coefficient: z is in units of 1 / H turns
                auto torus = [&](double v, int r) -> T {
                    if constexpr (S::kLvl1)
                        return turns_to_torus32(v * (fft512::scale(fft512::first_roots(), r) / H));
                    else
                        return double_to_torus<T>(v * (kTorusScale<T> / H));
                };
                if (more) {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const T lo = torus(z[r].x, r), hi = torus(z[r].y, r);
#pragma unroll
                        for (int p = 0; p < S::WORDS / R; p++) {
                            words[p * R + r] = pack(lo, hi, 0, p);
#pragma unroll
                            for (int q = 1; q < S::QW; q++)
                                reinterpret_cast<uint32_t*>(buf(slot, j, q * S::DPW))[(p * R + r) * 64 + lane] =
                                    pack(lo, hi, q, p);
                        }
                    }
                }
                else {
                    T* const res = reinterpret_cast<T*>(mine);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        res[lane + 64 * r] = torus(z[r].x, r);
                        res[lane + 64 * r + H] = torus(z[r].y, r);
                    }
                    wave_lds_sync();
                }
            }
            if (live && rooter && more) put(roots);
            if (more) {
                __syncthreads();  // next digits and roots are ready
                if (live && qi > 0) {
#pragma unroll
                    for (int w = 0; w < S::WORDS; w++)
                        words[w] = reinterpret_cast<const uint32_t*>(mine)[w * 64 + lane];
                    wave_lds_sync();
                }
            }
        }
    }
};

// SampleExtractIndex<0> of one component (as sample_extract_store), or the
// component itself, by one wave from its N coefficients in LDS.
template <class P>
__device__ __forceinline__ void pw_store(const typename P::T* c, int j, int lane, bool trlwe,
                                         typename P::T* out)
{
    using T = typename P::T;
    constexpr int N = P::n;
    if (trlwe) {
        for (int i = lane; i < N; i += 64) out[j * N + i] = c[i];
    }
    else if (j == 0) {
        for (int i = lane; i < N; i += 64)
            out[i] = i == 0 ? c[0] : static_cast<T>(0 - c[N - i]);
    }
    else if (lane == 0) {
        out[N] = c[0];
    }
}

}  // namespace cufhe_amd
