// Blind rotation with the digit transforms of a job spread over several waves
// and the multiply-accumulate split over all waves by spectrum bins: the key
// bundle at lvl1 and lvl2, CMUX keys (one TRGSW per key bit) at lvl1.
//
// Arithmetic: br_fft.hpp's steps (reference
// include/gatebootstrapping_gpu.cuh:895-1033 AccumulateKeyBundle, :69-221
// Accumulate, and :1335-1429 the drivers). At lvl2 operation for operation, so
// the outputs are bit-identical to k_br_fft. At lvl1 the external product is an
// integer that FP64 leaves within a small fraction of a unit, so any order of
// operations rounds to the same words: there the transforms are fft512.hpp's and
// X^(a0+a1) is the product of X^a0 and X^a1. With uniform keys and digits the
// bundle's product lies 0.0103 units rms from its integer, 0.059 at most over
// 61,440 coefficients (radix-8 transforms and the table's X^(a0+a1): 0.0122 and
// 0.070).
//
// A step has three phases, each ended by a workgroup barrier:
//  1. forward: wave (job, component j, qi) turns its DPW digit polynomials
//     into spectra, each in an LDS buffer that is the transform's scratch too;
//  2. multiply-accumulate: every wave takes R/W registers' worth of bins
//     (64 bins each) of all jobs. A key value is loaded from L2 by one wave,
//     straight into VGPRs, and used for every job: there is no key ring in LDS
//     and no barrier inside the phase. A lane reads the digit spectra at its
//     bins and writes the two output spectra over two of them (no other lane
//     touches those bins);
//  3. inverse: wave qi = 0 of (job, j) transforms component j's output back,
//     rounds, and hands the next digits to its partner waves through their idle
//     buffers; a partner (or the wave itself) prepares the next step's roots.
//     With CMUX keys it adds to the accumulator it keeps and publishes that in
//     LDS, where phase 1 reads it rotated.
// What bounds it: FP64 issue and LDS traffic, about equally, over the whole
// CU. (An LDS KiB costs a CU 5.7 ns written and 3.2 ns read at two waves per
// SIMD, a wave's FP64 instruction 0.5 ns; FP64 MFMA runs on the same pipe as
// the vector FMAs.) At lvl2 phase 2 also moves 786 KB of key a step through the
// CU's vector loads, which reach about 46 B/cycle.
#pragma once

#include "br_fft.hpp"
#include "fft512.hpp"

namespace cufhe_amd {

// J jobs per workgroup; DPW digit polynomials per wave; PF key blocks (three
// values) are in flight per lane.
template <class P_, int J_, int DPW_, int PF_, int HELP_ = 0, bool KB_ = true>
struct PwShape {
    using P = P_;
    using T = typename P::T;
    static constexpr int N = P::n, H = N / 2, R = H / 64, G = R / 8, L = P::l;
    static constexpr bool kLvl1 = sizeof(T) == 4;
    static constexpr int J = J_, DPW = DPW_, PF = PF_;
    static constexpr int QW = L / DPW;                // digit waves per component
    static constexpr int WPJ = 2 * QW, FW = J * WPJ;  // transform waves
    static constexpr int HELP = HELP_;                // waves of phase 2 only, and the roots
    static constexpr int W = FW + HELP, NT = 64 * W;
    static constexpr int BPL = R / W;                 // registers (64-bin groups) per wave in phase 2
    static constexpr int BLK = L * 4;                 // key blocks per register
    static constexpr int NB = BPL * BLK;              // key blocks
    static constexpr bool KB = KB_;
    static constexpr int NM = KB ? 3 : 1;  // key values of a block: the bundle's members
    static constexpr int STEPS = KB ? lvl0param::n / 2 : lvl0param::n;
    // root sets in LDS: lvl1 forms X^(a0+a1) as a product, lvl2 reads it from the table
    static constexpr int NX = kLvl1 ? 2 : 3;
    // digit words per lane: lvl1 one for both digits of two coefficients, lvl2
    // one for three digits of a coefficient
    static constexpr int WORDS = kLvl1 ? R : 2 * R;
    static constexpr bool kPrio = J > 1;  // several waves per SIMD meet at the barriers
    // all key blocks of a step in flight before phase 2 (else PF ahead, rolling)
    static constexpr bool kFull = PF == NB;
    // the roots of a job in the idle ends of its digit 1 buffers instead of an array
    static constexpr bool kTail = KB && kLvl1 && QW == 2 && HELP == 0;
    static constexpr bool kBase = KB && !kTail;
    static constexpr int TAB = kLvl1 ? fft512::kTabWords : 3 * 64;
    static_assert(QW * DPW == L, "shape");
    static_assert(kLvl1 ? L == 2 && P::Bgbit == 8 : DPW == 1 && L == 4 && P::Bgbit == 10, "digit words");
    static_assert(KB || kLvl1, "CMUX keys: lvl1");
    static_assert(HELP == 0 || HELP >= 2 * J, "two root waves per job");
    static_assert(!kFull || kLvl1, "the next step's keys are loaded in fft512's hooks");
    static_assert(BPL * W == R && NB % PF == 0, "even split");
};

template <class S>
struct PwShared {
    cplx buf[S::J * 2 * S::L][fft_stage::kScratchPad(S::H)];  // [(job * L + digit) * 2 + j]
    cplx base[S::kBase ? S::J : 1][S::NX][S::G][S::kBase ? 64 : 1];  // E[a (1 - 4 kb)] of a0, a1 (, a0 + a1)
    cplx tab[S::TAB];                                          // transform tables
    uint32_t a[S::J][S::NX];
    typename S::T acc[S::KB ? 1 : S::J][2][S::KB ? 1 : S::N];  // CMUX keys: the accumulators
};

// The lvl0 mask of a job: load(i) starts a coefficient on its way, value()
// mod-switches it to [0, 2N) (wave-uniform) a step later, so no wave waits for
// the load. ca * in0 + cb * in1 in global memory (in1 may be null), or words
// in LDS.
struct PwMask {
    const uint32_t* in0;
    const uint32_t* in1;
    uint32_t ca, cb;
    struct Raw {
        uint32_t x, y;
    };
    __device__ __forceinline__ Raw load(int i) const { return Raw{in0[i], in1 ? in1[i] : 0u}; }
    __device__ __forceinline__ uint32_t sum(Raw r) const { return ca * r.x + cb * r.y; }
    template <class P>
    __device__ __forceinline__ uint32_t value(Raw r) const
    {
        return __builtin_amdgcn_readfirstlane(mod_switch<P>(sum(r) + kMaskRound<P>));
    }
    // the rotation by the body (offset added)
    template <class P>
    __device__ __forceinline__ uint32_t body(uint32_t offset) const
    {
        return __builtin_amdgcn_readfirstlane(2 * P::n -
                                              mod_switch<P>(sum(load(lvl0param::n)) + offset));
    }
};

template <class S>
struct PwWave {
    using P = typename S::P;
    using T = typename S::T;
    static constexpr int N = S::N, H = S::H, R = S::R, L = S::L;
    static constexpr int kPer = S::WORDS / R;  // words of a coefficient pair
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
        return sm.buf[(s * L + ql) * 2 + comp];
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

    // Digit words of coefficients lo (r) and hi (R + r) for the wave qi = 0
    // (own) and for its partners. The digits are fields of c + offset less half
    // their range; with each field's top bit flipped they read as signed.
    // lvl1: both digits are the bytes 3 and 2, one word for two coefficients.
    // lvl2: four fields of 10 bits; the high word holds digits 0-2, bits 24-55
    // hold digits 1-3.
    struct Words {
        uint32_t own[2], partner[2];
    };
    __device__ __forceinline__ static Words pack(T lo, T hi)
    {
        if constexpr (S::kLvl1) {
            const uint32_t a = lo + Gadget<P>::kOffset, b = hi + Gadget<P>::kOffset;
            const uint32_t w = ((a >> 16) | (b & 0xffff0000u)) ^ 0x80808080u;
            return Words{{w, 0u}, {w, 0u}};
        }
        else {
            constexpr uint64_t flip = (1ull << 63) | (1ull << 53) | (1ull << 43) | (1ull << 33);
            const uint64_t a = (lo + Gadget<P>::kOffset) ^ flip, b = (hi + Gadget<P>::kOffset) ^ flip;
            return Words{{static_cast<uint32_t>(a >> 32), static_cast<uint32_t>(b >> 32)},
                         {static_cast<uint32_t>(a >> 24), static_cast<uint32_t>(b >> 24)}};
        }
    }
    // folded digit m of this wave (gadget digit qi DPW + m) at register r
    __device__ __forceinline__ cplx digits(int r, int m) const
    {
        const int q = qi * S::DPW + m;
        auto field = [](uint32_t w, int at, int bits) {
            return static_cast<double>(static_cast<int32_t>(__builtin_amdgcn_sbfe(w, at, bits)));
        };
        if constexpr (S::kLvl1) {
            return cplx{field(words[r], 8 * (1 - q), 8), field(words[r], 24 - 8 * q, 8)};
        }
        else {
            const int at = qi == 0 ? 22 - 10 * q : 30 - 10 * q;
            return cplx{field(words[2 * r], at, 10), field(words[2 * r + 1], at, 10)};
        }
    }
    __device__ __forceinline__ void init_digits(uint32_t bar, T mu)
    {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i0 = lane + 64 * r;
            const T lo = j == 0 ? T(0) : test_vector_coef<P>(i0, bar, mu);
            const T hi = j == 0 ? T(0) : test_vector_coef<P>(i0 + H, bar, mu);
            const Words v = pack(lo, hi);
#pragma unroll
            for (int k = 0; k < kPer; k++) words[kPer * r + k] = qi == 0 ? v.own[k] : v.partner[k];
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

    // Key block b of a step: register dd, digit, component, output column; its
    // three bundle members.
    struct KeyBlk {
        cplx k[S::NM];
    };
    __device__ __forceinline__ KeyBlk load_key(int step, int b, int d0) const
    {
        constexpr size_t TS = kTrgswFourier<P>;
        const int dd = b / S::BLK, ql = (b % S::BLK) / 4, comp = (b / 2) & 1, col = b & 1;
        // wave-uniform address (SGPRs) plus the lane's 32-bit byte offset
        const uint32_t st = __builtin_amdgcn_readfirstlane(step);
        const uint32_t in_step = __builtin_amdgcn_readfirstlane(
            ((comp * L + ql) * 2 + col) * H + (d0 + dd) * 64);
        const uint64_t u = reinterpret_cast<uint64_t>(K.bk + st * (S::NM * TS) + in_step);
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
        KeyBlk v;
#pragma unroll
        for (int e = 0; e < S::NM; e++) v.k[e] = at(e);
        return v;
    }

    // lvl2 batches: reads a word of every 128-byte line of a step's key, so that
    // the key loads of that step find them in L2. `groups` workgroups, the first of
    // the grid, rotate in step; those of an XCD (one in eight) share the lines over
    // their four waves that are idle in phase 3. The key outgrows the caches next
    // to the key-switching key, and a rotation that waits for it took 5.3 ms for 64
    // to 256 jobs; 4.3 so (2048-gate mix 47.6 -> 42.1 ms). Fewer than 25 workgroups
    // would need more than six loads a lane, which phase 3 does not hide (8 jobs
    // 5.7 -> 7.5 ms), and read no lines ahead.
    __device__ __forceinline__ void touch_key(int step, uint32_t groups) const
    {
        constexpr uint32_t kStep = S::NM * kTrgswFourier<P> * sizeof(cplx), kLine = 128;
        const uint32_t waves = (groups + 7) / 8 * 4, mine = blockIdx.x / 8 * 4 + (qi - 2) * 2 + j;
        if (waves * 64 * 6 * kLine < kStep) return;
        const char* const p = reinterpret_cast<const char*>(K.bk) + static_cast<size_t>(step) * kStep;
        uint32_t x = 0;
#pragma unroll 6
        for (uint32_t at = (mine * 64 + lane) * kLine; at < kStep; at += waves * 64 * kLine)
            x ^= *reinterpret_cast<const uint32_t*>(p + at);
        asm volatile("" ::"v"(x));
    }

    // The rotation of the workgroup's jobs. mask: that of this wave's job, bar:
    // its body's rotation. live: whether this wave's job exists. At the end the
    // buffer of (job, j, digit 0) holds the N coefficients of component j (visible
    // to the wave with qi = 0). TOUCH: touch_key ahead, with `groups`.
    template <bool TOUCH = false>
    __device__ __forceinline__ void rotate(bool live, uint32_t bar, T mu, const PwMask& mask,
                                           uint32_t groups = 1)
    {
        constexpr int PF = S::PF, NB = S::NB;
        const int d0 = wave * S::BPL;
        const bool fft = live && qi >= 0;
        cplx* const mine = buf(slot, j, (qi < 0 ? 0 : qi) * S::DPW);
        const fft512::Slots slots = fft512::Slots::of(lane);
        PwMask::Raw na0{0, 0}, na1{0, 0};  // the next step's mask coefficients
        T acc[S::KB ? 1 : 2 * R];  // CMUX keys: this wave's component
        if constexpr (S::KB) {
            if (fft) init_digits(bar, mu);
        }
        else {
            if (fft && qi == 0) {
#pragma unroll
                for (int r = 0; r < 2 * R; r++) {
                    const int i = AccStore<P>::coef_index(r, lane);
                    acc[r] = j == 0 ? T(0) : test_vector_coef<P>(i, bar, mu);
                    sm.acc[slot][j][i] = acc[r];
                }
            }
            if (fft) na0 = mask.load(0);
        }
        cplx tail_root;  // kTail: the next root until its place is free
        if (S::KB && live && rooter) {
            const Gathered first =
                gather(mask.value<P>(mask.load(0)), mask.value<P>(mask.load(1)));
            put(first);
            tail_root = first.v[0][0];
            na0 = mask.load(2);
            na1 = mask.load(3);
        }
        auto next_mask = [&](int it) {
            if (it + 2 < S::STEPS) {
                na0 = mask.load(2 * it + 4);
                na1 = mask.load(2 * it + 5);
            }
        };
        KeyBlk kv[PF];
        // full prefetch: transform waves that run the inverse load during the
        // next forward transform, the others during the inverse phase
        const bool early = !S::kFull || qi != 0;
        if (early) {
#pragma unroll
            for (int b = 0; b < PF; b++) kv[b] = load_key(0, b, d0);
        }
        __syncthreads();  // the first roots
#pragma unroll 1
        for (int it = 0; it < S::STEPS; it++) {
            // the last blocks of a step prefetch the next step's first ones
            const int next = it + 1 < S::STEPS ? it + 1 : it;
            // W_8^(a d) of this step: scalar loads, at lvl1 long before their use
            // (at lvl2 the transforms need the SGPRs)
            cplx w8[S::BPL][S::J][S::NX];
            auto load_w8 = [&]() {
#pragma unroll
                for (int jl = 0; jl < S::J; jl++)
#pragma unroll
                    for (int m = 0; m < S::NX; m++) {
                        const uint32_t a = __builtin_amdgcn_readfirstlane(sm.a[jl][m]);
#pragma unroll
                        for (int dd = 0; dd < S::BPL; dd++) {
                            const int e = (a * static_cast<uint32_t>(d0 + dd)) & 7u;
                            w8[dd][jl][m] = cplx{kW8[e][0], kW8[e][1]};
                        }
                    }
            };
            if constexpr (S::KB && S::kLvl1) load_w8();
            const bool more = it + 1 < S::STEPS;
            Gathered roots;
            if (S::KB && S::HELP && live && rooter && more) {
                // helpers gather the next step's roots while the others transform
                roots = gather(mask.value<P>(na0), mask.value<P>(na1));
                next_mask(it);
            }
            cplx s[S::BPL][S::J][2];
#pragma unroll
            for (int dd = 0; dd < S::BPL; dd++)
#pragma unroll
                for (int jl = 0; jl < S::J; jl++) s[dd][jl][0] = s[dd][jl][1] = cplx{0.0, 0.0};
            if constexpr (!S::KB) {
                // digits of (X^a - 1) acc
                if (fft) {
                    const uint32_t a = mask.value<P>(na0);
                    if (more) na0 = mask.load(it + 1);
                    const T* const src = sm.acc[slot][j];
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const int i = lane + 64 * r;
                        // X^a acc at i: acc[(i - a) mod N], negated where bit
                        // log N of i - a (mod 2N) is set
                        auto rotated = [&](int k) {
                            const uint32_t u = static_cast<uint32_t>(k) - a;
                            const uint32_t neg = 0u - ((u >> P::nbit) & 1u);
                            return (static_cast<uint32_t>(src[u & (N - 1)]) ^ neg) - neg;
                        };
                        const Words v = pack(static_cast<T>(rotated(i)) - src[i],
                                             static_cast<T>(rotated(i + H)) - src[i + H]);
                        words[r] = v.own[0];
                    }
                }
            }
            if (fft) {
                if constexpr (S::kLvl1) {
                    cplx z[S::DPW][8];
                    cplx* zb[S::DPW];
#pragma unroll
                    for (int m = 0; m < S::DPW; m++) {
                        zb[m] = buf(slot, j, qi * S::DPW + m);
#pragma unroll
                        for (int r = 0; r < 8; r++) z[m][r] = digits(r, m);
                    }
                    // a third of the key blocks behind each stage's stores: the
                    // vector memory queue takes 16 cycles a load and CU
                    fft512::forward<S::DPW, S::kPrio>(z, zb, tables(), slots, lane, [&](int part) {
                        if constexpr (S::kFull)
                            if (qi == 0 || S::QW == 1)
#pragma unroll
                                for (int b = 0; b < PF; b++)
                                    if (b * 3 / PF == part) kv[b] = load_key(it, b, d0);
                    });
                }
                else {
                    using namespace fft_stage;
                    cplx z[R];
#pragma unroll
                    for (int r = 0; r < R; r++) z[r] = digits(r, 0);
                    const FFTTables tb = lvl2_tables();
                    wave_prio<true>(3);
#pragma unroll
                    for (int r = 1; r < R; r++) z[r] = cmul(z[r], cr(r));
                    fwd_a_dft<R>(z, tb, lane);
                    t1_store<R>(z, mine, lane);
                    wave_lds_sync();
                    t1_load<R>(z, mine, lane);
                    wave_lds_sync();
                    wave_prio<true>(2);
                    fwd_b<R>(z, tb, lane);
                    t2_store_cx<R>(z, mine, lane);
                    wave_lds_sync();
                    t2_load_xc<R>(z, mine, lane);
                    wave_lds_sync();
                    wave_prio<true>(1);
                    fwd_c<R>(z);
                    wave_prio<true>(0);
#pragma unroll
                    for (int d = 0; d < R; d++) lds_store(&mine[d * 64 + lane], z[d]);
                }
            }
            if constexpr (S::kTail)
                if (live && rooter) lds_store(&mine[H + lane], tail_root);
            if (!fft && S::kFull && !early) {
                // no job: the wave still multiplies for the others
#pragma unroll
                for (int b = 0; b < PF; b++) kv[b] = load_key(it, b, d0);
            }
            // X^a - 1 at this wave's bins; the roots were published a barrier ago
            cplx x[S::BPL][S::J][3];
            auto make_x = [&]() {
                if constexpr (!S::kLvl1) load_w8();
#pragma unroll
                for (int dd = 0; dd < S::BPL; dd++)
#pragma unroll
                    for (int jl = 0; jl < S::J; jl++) {
                        cplx(&xx)[3] = x[dd][jl];
#pragma unroll
                        for (int m = 0; m < S::NX; m++)
                            xx[m] = cmul(lds_load(&root(jl, m, (d0 + dd) >> 3)[lane]), w8[dd][jl][m]);
                        if constexpr (S::NX == 2) xx[2] = cmul(xx[0], xx[1]);
#pragma unroll
                        for (int m = 0; m < 3; m++) xx[m].x -= 1.0;
                    }
            };
            // with helper waves after the barrier: before it, their key
            // loads were waited for there (one gate 1.35 against 1.25 ms)
            if constexpr (S::kBase && !S::HELP) make_x();
            __syncthreads();  // digit spectra are in LDS
            if constexpr (S::kTail || (S::kBase && S::HELP)) make_x();
            // the spectra of a (digit, component) are loaded while the one
            // before it is multiplied
            constexpr int DN = S::BPL * L * 2;
            cplx D[2][S::J];
            auto load_d = [&](int n, cplx(&dst)[S::J]) {
                const int dd = n / (2 * L), ql = (n / 2) % L, comp = n & 1;
#pragma unroll
                for (int jl = 0; jl < S::J; jl++)
                    dst[jl] = lds_load(&buf(jl, comp, ql)[(d0 + dd) * 64 + lane]);
            };
            load_d(0, D[0]);
            wave_prio<S::kPrio>(3);
#pragma unroll
            for (int dd = 0; dd < S::BPL; dd++) {
#pragma unroll
                for (int ql = 0; ql < L; ql++) {
                    const double hq = ldexp(1.0, -static_cast<int>((ql + 1) * P::Bgbit));
#pragma unroll
                    for (int comp = 0; comp < 2; comp++) {
                        const int n = (dd * L + ql) * 2 + comp;
                        if (n + 1 < DN) load_d(n + 1, D[(n + 1) & 1]);
                        if (n == DN / 4) wave_prio<S::kPrio>(2);
                        if (n == DN / 2) wave_prio<S::kPrio>(1);
                        if (n == DN * 3 / 4) wave_prio<S::kPrio>(0);
#pragma unroll
                        for (int col = 0; col < 2; col++) {
                            const int i = dd * S::BLK + ql * 4 + comp * 2 + col;
                            const KeyBlk cur = kv[i % PF];
                            if constexpr (!S::kFull)
                                kv[i % PF] = i + PF < NB ? load_key(it, i + PF, d0) : load_key(next, i + PF - NB, d0);
#pragma unroll
                            for (int jl = 0; jl < S::J; jl++) {
                                cplx k = cur.k[0];
                                if constexpr (S::KB) {
                                    k = cplx{comp == col ? hq : 0.0, 0.0};
                                    cmac(k, cur.k[2], x[dd][jl][1]);
                                    cmac(k, cur.k[1], x[dd][jl][0]);
                                    cmac(k, cur.k[0], x[dd][jl][2]);
                                }
                                cmac(s[dd][jl][col], D[n & 1][jl], k);
                            }
                            // the loads of later blocks stay behind this block's products
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
#pragma unroll
            for (int dd = 0; dd < S::BPL; dd++)
#pragma unroll
                for (int jl = 0; jl < S::J; jl++)
#pragma unroll
                    for (int col = 0; col < 2; col++)
                        lds_store(&buf(jl, col, 0)[(d0 + dd) * 64 + lane], s[dd][jl][col]);
            __syncthreads();  // output spectra are in the digit 0 buffers
            if (S::KB && S::HELP == 0 && live && rooter && more) {
                if constexpr (!S::kLvl1) {  // an idle partner wave, short of VGPRs
                    na0 = mask.load(2 * it + 2);
                    na1 = mask.load(2 * it + 3);
                }
                roots = gather(mask.value<P>(na0), mask.value<P>(na1));
                if constexpr (S::kLvl1) next_mask(it);
            }
            // (behind the roots' loads: they return in order)
            if (S::kFull && early) {
#pragma unroll
                for (int b = 0; b < PF; b++) kv[b] = load_key(next, b, d0);
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
                    t2_store_xc<R>(z, mine, lane);
                    wave_lds_sync();
                    t2_load_cx<R>(z, mine, lane);
                    wave_lds_sync();
                    inv_b<R>(z, tb, lane);
                    t1_store_inv<R>(z, mine, lane);
                    wave_lds_sync();
                    t1_load_inv<R>(z, mine, lane);
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
                if constexpr (!S::KB) {
                    T* const res = more ? sm.acc[slot][j] : reinterpret_cast<T*>(mine);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        acc[r] += torus(z[r].x, r);
                        acc[R + r] += torus(z[r].y, r);
                        res[lane + 64 * r] = acc[r];
                        res[lane + 64 * r + H] = acc[R + r];
                    }
                    wave_lds_sync();
                }
                else if (more) {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const T lo = torus(z[r].x, r), hi = torus(z[r].y, r);
                        const Words v = pack(lo, hi);
#pragma unroll
                        for (int k = 0; k < kPer; k++) {
                            words[kPer * r + k] = v.own[k];
#pragma unroll
                            for (int q = 1; q < S::QW; q++)
                                reinterpret_cast<uint32_t*>(buf(slot, j, q * S::DPW))[(kPer * r + k) * 64 + lane] =
                                    v.partner[k];
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
            if constexpr (TOUCH)
                if (more && qi > 1) touch_key(next, groups);
            if (S::KB && live && rooter && more) {
                put(roots);
                if constexpr (S::kTail) tail_root = roots.v[0][0];
            }
            if (more) {
                __syncthreads();  // next digits and roots are ready
                if (S::KB && live && qi > 0) {
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
