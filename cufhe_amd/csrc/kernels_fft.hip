// FFT-backend kernels: key conversion, batched blind rotation, plain
// per-gate kernels, key switching, MUX combine, and FFNT entry points.
#include "br_fft.hpp"
#include "br_fft_pw.hpp"
#include "keyswitch.hpp"
#include "launch.hpp"
#include "launch_rules.hpp"

namespace cufhe_amd {

constexpr int kTlwe0Pad = 640;  // lvl0 TLWE (637 words) padded in LDS

// ---------------------------------------------------------------------------
// Polynomial -> Fourier spectra. One wave per polynomial.
// Reference src/bootstrap_gpu.cu:59-112 (__TRGSW2FFT__): signed torus value
// * 2^-w, fold, twist, forward FFT. INTEGER=true skips the 2^-w scaling and
// reads int32 inputs (used for X^a - 1 and test polynomials).
template <class P, bool INTEGER>
__global__ __launch_bounds__(256) void k_to_fourier(cplx* out, const void* in, int npolys,
                                                    FourierKeys<P> K)
{
    using T = typename P::T;
    using ST = std::make_signed_t<T>;
    constexpr int N = P::n, H = N / 2, R = H / 64;
    __shared__ cplx sc[4][H];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int poly = blockIdx.x * 4 + wave;
    if (poly >= npolys) return;  // no workgroup barriers below
    cplx z[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int m = lane + 64 * r;
        double re, im;
        if constexpr (INTEGER) {
            const int32_t* p = static_cast<const int32_t*>(in) + static_cast<size_t>(poly) * N;
            re = static_cast<double>(p[m]);
            im = static_cast<double>(p[m + H]);
        }
        else {
            const T* p = static_cast<const T*>(in) + static_cast<size_t>(poly) * N;
            constexpr double s = 1.0 / kTorusScale<T>;
            re = static_cast<double>(static_cast<ST>(p[m])) * s;
            im = static_cast<double>(static_cast<ST>(p[m + H])) * s;
        }
        z[r] = cplx{re, im};
    }
    fft_forward<H>(z, sc[wave], K.fft);
#pragma unroll
    for (int d = 0; d < R; d++) out[static_cast<size_t>(poly) * H + d * 64 + lane] = z[d];
}

// X^a - 1 polynomials for a in [0, 2N) (reference src/ntt_small_modulus.cu
// :928-981 XaittGen): coefficient 0 is -1, coefficient a mod N gets +1
// (a < N) or -1 (a >= N).
template <class P>
__global__ void k_xai_poly(int32_t* out)
{
    constexpr int N = P::n;
    const int a = blockIdx.x;
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
        int32_t v = (i == 0) ? -1 : 0;
        if (i == (a & (N - 1))) v += (a < N) ? 1 : -1;
        out[static_cast<size_t>(a) * N + i] = v;
    }
}

// Spectra -> real polynomial (inverse FFT, untwist incl. 1/H), as doubles.
template <class P>
__global__ __launch_bounds__(256) void k_from_fourier(double* out, const cplx* in, int npolys,
                                                      FourierKeys<P> K)
{
    constexpr int N = P::n, H = N / 2, R = H / 64;
    __shared__ cplx sc[4][H];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int poly = blockIdx.x * 4 + wave;
    if (poly >= npolys) return;
    cplx z[R];
#pragma unroll
    for (int d = 0; d < R; d++) z[d] = in[static_cast<size_t>(poly) * H + d * 64 + lane];
    fft_inverse<H>(z, sc[wave], K.fft);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int m = lane + 64 * r;
        const cplx v = cscale(z[r], 1.0 / H);
        out[static_cast<size_t>(poly) * N + m] = v.x;
        out[static_cast<size_t>(poly) * N + m + H] = v.y;
    }
}

// ---------------------------------------------------------------------------
// Batched lvl2 rotation with two waves per job (CMUX keys; the key bundle with
// two jobs per workgroup): C jobs per workgroup. The workgroups walk the job
// groups with a grid stride, so a grid that fits on the device at once keeps
// every workgroup on the same rotation step: their key reads then meet in L2
// instead of drifting apart as later workgroups start when earlier ones finish.
template <bool KB, int C>
__global__ __launch_bounds__(128 * C, C > 1 ? 1 : 3) void k_br_fft(const BrJob* __restrict__ jobs,
                                                                   int njobs, uint64_t mu,
                                                                   FourierKeys<lvl2param> K)
{
    using P = lvl2param;
    using T = uint64_t;
    constexpr int N = P::n, H = N / 2, n0 = lvl0param::n;
    constexpr int NB = BrShape<P>::NB;
    __shared__ cplx sh_spec[2 * C][NB * H];
    __shared__ uint32_t sh_tl0[C][kTlwe0Pad];
    __shared__ T sh_coef[2 * C][N];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = wave >> 1, j = wave & 1;
    const int ngroups = (njobs + C - 1) / C;
    for (int grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const int raw = grp * C + slot;
        const bool live = raw < njobs;
        const BrJob jb = jobs[live ? raw : njobs - 1];
        // the previous group's rotation has finished reading sh_tl0
        __syncthreads();
        for (int i = threadIdx.x & 127; i <= n0; i += 128) {
            uint32_t v = static_cast<uint32_t>(jb.ca) * jb.in0[i];
            if (jb.in1) v += static_cast<uint32_t>(jb.cb) * jb.in1[i];
            if (i == n0) v += jb.offset;
            sh_tl0[slot][i] = v;
        }
        __syncthreads();
        AccStore<P> acc;
        acc.lds = sh_coef[wave];
        blind_rotate_fft<P, KB>(sh_tl0[slot], mu, acc, j, sh_spec[wave], sh_spec[wave ^ 1], K);
        if (live) {
            if (jb.flags & kBrOutTrlwe)
                trlwe_store<P>(acc, j, static_cast<T*>(jb.out));
            else
                sample_extract_store<P>(acc, j, static_cast<T*>(jb.out));
        }
    }
}

// Workgroups of k_br_fft<KB, C> resident on the device at once (0 if the
// runtime cannot tell), cached per instance.
template <bool KB, int C>
static int br_fft_resident_groups()
{
    static int cached = -1;
    int v = __atomic_load_n(&cached, __ATOMIC_RELAXED);
    if (v < 0) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_br_fft<KB, C>, 128 * C, 0) !=
                hipSuccess ||
            per_cu < 0)
            per_cu = 0;
        v = per_cu * device_cu_count();
        __atomic_store_n(&cached, v, __ATOMIC_RELAXED);
    }
    return v;
}

// ---------------------------------------------------------------------------
// Batched key-bundle rotation, one wave per digit polynomial (br_fft_pw.hpp):
// S::J jobs per workgroup; the workgroups walk the job groups with a grid
// stride.
template <class S, int WPE>
__global__ __launch_bounds__(S::NT, WPE) void k_br_fft_pw(const BrJob* __restrict__ jobs, int njobs,
                                                          typename S::T mu,
                                                          FourierKeys<typename S::P> K)
{
    using P = typename S::P;
    using T = typename S::T;
    __shared__ PwShared<S> sm;
    PwWave<S> w(sm, K, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63);
    w.load_tables(threadIdx.x);
    __syncthreads();
    const int ngroups = (njobs + S::J - 1) / S::J;
    for (int grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const int raw = grp * S::J + w.slot;
        const bool live = raw < njobs;
        const BrJob jb = jobs[live ? raw : njobs - 1];
        const PwMask mask{jb.in0, jb.in1, static_cast<uint32_t>(jb.ca), static_cast<uint32_t>(jb.cb)};
        if constexpr (S::kLvl1) {
            w.rotate(live, mask.body<P>(jb.offset), mu, mask);
        }
        else {
            // the workgroups that have a group in this round
            const int left = ngroups - (grp - static_cast<int>(blockIdx.x));
            w.template rotate<true>(live, mask.body<P>(jb.offset), mu, mask,
                                    min(static_cast<int>(gridDim.x), left));
        }
        if (live && w.qi == 0)
            pw_store<P>(reinterpret_cast<const T*>(w.buf(w.slot, w.j, 0)), w.j, w.lane,
                        jb.flags & kBrOutTrlwe, static_cast<T*>(jb.out));
    }
}

// The lvl2 shape: eight waves, one digit polynomial each, two 64-bin groups of
// the products. Four key blocks (12 KiB) in flight a wave: the phase streams
// 786 KB of key through the CU's L2 path; eight spill.
using Lvl2Shape = PwShape<lvl2param, 1, 1, 4>;

// ---------------------------------------------------------------------------
// SampleExtract + key switch lvl1 -> lvl0 of n TRLWEs (reference SEIandKS,
// src/keyswitch_gpu.cu:61-68, include/keyswitch_gpu.cuh:52-123), one job per
// workgroup.
template <bool SUBSET>
__global__ __launch_bounds__(512) void k_se_ks_lvl10(uint32_t* out, const uint32_t* trlwe, int n,
                                                     const uint32_t* ksk)
{
    constexpr int N = lvl1param::n, n0 = lvl0param::n;
    __shared__ uint32_t tl[N + 4];
    __shared__ uint32_t sh_red[8 * (n0 + 1)];
    const int job = blockIdx.x;
    if (job >= n) return;  // whole workgroup
    const uint32_t* tr = trlwe + static_cast<size_t>(job) * 2 * N;
    for (int i = threadIdx.x; i <= N; i += 512)
        tl[i] = i == 0 ? tr[0] : (i < N ? 0u - tr[N - i] : tr[N]);
    __syncthreads();
    // the input coefficients split over the eight waves (a job's key switch
    // is a long dependent gather loop; eight shorter ones hide its latency)
    key_switch_waves<TFHEpp::lvl10param, SUBSET, 8>(out + static_cast<size_t>(job) * (n0 + 1), tl,
                                                    nullptr, 1, 0, 0u, ksk, sh_red,
                                                    __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                                                    threadIdx.x & 63);
}

// ---------------------------------------------------------------------------
// Plain per-gate form at lvl1 (reference src/bootstrap_gpu.cu:1223-1246,
// :1557-1672, :2069-2197, src/cufhe_gates_gpu.cu:198-511), one gate per
// workgroup of eight waves on br_fft_pw.hpp's rotation: four transform waves and four that
// help with the products and the roots (MUX/NMUX: two jobs of four transform
// waves). Same key switch and rotation as the batched form, so the outputs are
// the same words. One NAND of the lvl1 API took 3.80 ms with the rotation on a
// single wave and the others only streaming the key; now 1.25 ms (MUX 4.40 ->
// 1.84 ms).
template <bool KB, bool MUX>
using GateShape = PwShape<lvl1param, MUX ? 2 : 1, 1, 8, MUX ? 0 : 4, KB>;

// coefficient i of SampleExtractIndex<0> of job `job` (its components lie in
// the digit 0 buffers after rotate())
template <class S>
__device__ __forceinline__ uint32_t gate_sample(const PwWave<S>& w, int job, int i)
{
    const uint32_t* a = reinterpret_cast<const uint32_t*>(w.buf(job, 0, 0));
    if (i == S::N) return reinterpret_cast<const uint32_t*>(w.buf(job, 1, 0))[0];
    return i == 0 ? a[0] : 0u - a[S::N - i];
}

// lvl1 API (IKS then BR): MUX/NMUX run c + t - mu and -c + f - mu.
template <bool KB, bool MUX>
__global__ __launch_bounds__(512, 2) void k_gate_lvl1_pw(
    uint32_t* out, const uint32_t* in0, const uint32_t* in1, const uint32_t* inc, int32_t ca,
    int32_t cb, uint32_t offset, int32_t mux_sign, const uint32_t* ksk,
    FourierKeys<lvl1param> K)
{
    using P = lvl1param;
    using S = GateShape<KB, MUX>;
    static_assert(S::NT == 512, "eight waves");
    constexpr int N = P::n, n0 = lvl0param::n;
    constexpr uint32_t mu = static_cast<uint32_t>(P::μ);
    __shared__ PwShared<S> sm;
    __shared__ uint32_t sh_tl0[S::J][kTlwe0Pad];
    PwWave<S> w(sm, K, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63);
    w.load_tables(threadIdx.x);
    // key switch over all eight waves (MUX: four per rotation input), partial
    // sums in the transform buffers
    uint32_t* const red = reinterpret_cast<uint32_t*>(&sm.buf[0][0]);
    if constexpr (MUX) {
        const int job = w.wave >> 2;
        key_switch_waves<TFHEpp::lvl10param, false, 4>(
            sh_tl0[job], inc, job == 0 ? in1 : in0, job == 0 ? 1 : -1, 1, 0u - mu, ksk,
            red + job * 4 * (n0 + 1), w.wave & 3, w.lane);
    }
    else {
        key_switch_waves<TFHEpp::lvl10param, false, 8>(sh_tl0[0], in0, in1, ca, cb, offset, ksk,
                                                       red, w.wave, w.lane);
    }
    __syncthreads();
    const PwMask mask{sh_tl0[w.slot], nullptr, 1, 0};
    w.rotate(true, mask.body<P>(0), mu, mask);
    __syncthreads();
    for (int i = threadIdx.x; i <= N; i += S::NT) {
        uint32_t v = gate_sample(w, 0, i);
        if constexpr (MUX) {
            v += gate_sample(w, 1, i) + (i == N ? mu : 0u);
            if (mux_sign < 0) v = 0u - v;
        }
        out[i] = v;
    }
}

// lvl0 API (BR then IKS): the pre-added lvl0 inputs are mod-switched as they
// are read; the extracted samples wait in LDS for the key switch.
template <bool KB, bool MUX, bool SUBSET>
__global__ __launch_bounds__(512, 2) void k_gate_lvl01_pw(
    uint32_t* out, const uint32_t* in0, const uint32_t* in1, const uint32_t* inc, int32_t ca,
    int32_t cb, uint32_t offset, int32_t mux_sign, uint32_t tv_mu, const uint32_t* ksk,
    FourierKeys<lvl1param> K)
{
    using P = lvl1param;
    using S = GateShape<KB, MUX>;
    constexpr int N = P::n;
    constexpr uint32_t mu = static_cast<uint32_t>(P::μ);
    constexpr uint32_t mu0 = static_cast<uint32_t>(lvl0param::μ);
    __shared__ PwShared<S> sm;
    __shared__ uint32_t sh_res[S::J][N + 4];
    PwWave<S> w(sm, K, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63);
    w.load_tables(threadIdx.x);
    __syncthreads();
    const uint32_t* a = MUX ? inc : in0;
    const uint32_t* b = MUX ? (w.slot == 0 ? in1 : in0) : in1;
    const uint32_t sa = static_cast<uint32_t>(MUX ? (w.slot == 0 ? 1 : -1) : ca);
    const uint32_t sb = static_cast<uint32_t>(MUX ? 1 : cb);
    const uint32_t off = MUX ? 0u - mu0 : offset;
    const PwMask mask{a, b, sa, sb};
    w.rotate(true, mask.body<P>(off), tv_mu, mask);
    __syncthreads();
#pragma unroll
    for (int job = 0; job < S::J; job++)
        for (int i = threadIdx.x; i <= N; i += S::NT) sh_res[job][i] = gate_sample(w, job, i);
    __syncthreads();
    uint32_t* const red = reinterpret_cast<uint32_t*>(&sm.buf[0][0]);
    if constexpr (MUX)
        key_switch_waves<TFHEpp::lvl10param, SUBSET, 8>(out, sh_res[0], sh_res[1], mux_sign,
                                                        mux_sign, mux_sign > 0 ? mu : 0u - mu, ksk,
                                                        red, w.wave, w.lane);
    else
        key_switch_waves<TFHEpp::lvl10param, SUBSET, 8>(out, sh_res[0], nullptr, 1, 0, 0u, ksk,
                                                        red, w.wave, w.lane);
}

// ---------------------------------------------------------------------------
// Plain per-gate form, lvl02 API (BR-IKS order): lvl0 in, BR to lvl2
// (Torus64), SE, key switch lvl2 -> lvl0 (reference src/bootstrap_gpu.cu
// :1248-1273, :1305-1331, MUX :1949-2060). MUX runs its two rotations one
// after the other in the same wave pair (LDS holds one lvl2 job).
template <bool MUX>
__global__ __launch_bounds__(256, 1) void k_gate_lvl02_fft(
    uint32_t* out, const uint32_t* in0, const uint32_t* in1, const uint32_t* inc, int32_t ca,
    int32_t cb, uint32_t offset, int32_t mux_sign, const uint32_t* ksk,
    FourierKeys<lvl2param> K)
{
    using P = lvl2param;
    using T = uint64_t;
    constexpr int N = P::n, H = N / 2, n0 = lvl0param::n;
    constexpr T mu = static_cast<T>(P::μ);
    constexpr int NB = BrShape<P>::NB;
    __shared__ cplx sh_spec[2][NB * H];
    __shared__ T sh_coef[2][N];
    __shared__ uint32_t sh_tl0[kTlwe0Pad];
    __shared__ T sh_res[MUX ? 2 : 1][N + 8];
    // waves 0 and 1 rotate; waves 2 and 3 keep step through the rotation's
    // barriers and then join the key switch (four waves: one per SIMD, so
    // the rotating waves keep the whole register file)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = wave & 1;
    const int t = threadIdx.x & 127;
    const bool rotating = wave < 2;
    AccStore<P> acc;
    acc.lds = sh_coef[j];
#pragma unroll 1
    for (int pass = 0; pass < (MUX ? 2 : 1); pass++) {
        // MUX: pass 0 = c + t - mu, pass 1 = -c + f - mu
        const uint32_t* a = MUX ? inc : in0;
        const uint32_t* b = MUX ? (pass == 0 ? in1 : in0) : in1;
        const int32_t sa = MUX ? (pass == 0 ? 1 : -1) : ca;
        const int32_t sb = MUX ? 1 : cb;
        const uint32_t off = MUX ? 0u - static_cast<uint32_t>(lvl0param::μ) : offset;
        __syncthreads();
        if (rotating) {
            for (int i = t; i <= n0; i += 128) {
                uint32_t v = static_cast<uint32_t>(sa) * a[i] + static_cast<uint32_t>(sb) * b[i];
                if (i == n0) v += off;
                sh_tl0[i] = v;
            }
        }
        __syncthreads();
        if (rotating) {
            blind_rotate_fft<P, false>(sh_tl0, mu, acc, j, sh_spec[j], sh_spec[j ^ 1], K);
            sample_extract_store<P>(acc, j, sh_res[pass]);
        }
        else {
            blind_rotate_ghost<P, false>(K);
        }
    }
    __syncthreads();
    // partial sums of the key switch in the (now free) transform scratch
    uint32_t* const red = reinterpret_cast<uint32_t*>(&sh_spec[0][0]);
    if constexpr (MUX) {
        key_switch_waves<TFHEpp::lvl20param, false, 4>(out, sh_res[0], sh_res[1], mux_sign,
                                                       mux_sign, mux_sign > 0 ? mu : 0 - mu, ksk,
                                                       red, wave, threadIdx.x & 63);
    }
    else {
        key_switch_waves<TFHEpp::lvl20param, false, 4>(out, sh_res[0], nullptr, 1, 0, 0, ksk, red,
                                                       wave, threadIdx.x & 63);
    }
}

// The same with the key bundle on br_fft_pw.hpp's rotation (eight waves). MUX
// runs its two rotations one after the other (the LDS holds one lvl2 job); the
// first one's sample waits in registers.
template <bool MUX>
__global__ __launch_bounds__(512, 2) void k_gate_lvl02_pw(
    uint32_t* out, const uint32_t* in0, const uint32_t* in1, const uint32_t* inc, int32_t ca,
    int32_t cb, uint32_t offset, int32_t mux_sign, const uint32_t* ksk,
    FourierKeys<lvl2param> K)
{
    using P = lvl2param;
    using T = uint64_t;
    using S = Lvl2Shape;
    constexpr int N = P::n, n0 = lvl0param::n, PER = N / S::NT;
    constexpr T mu = static_cast<T>(P::μ);
    constexpr uint32_t mu0 = static_cast<uint32_t>(lvl0param::μ);
    static_assert(S::NT == 512, "eight waves");
    __shared__ PwShared<S> sm;
    PwWave<S> w(sm, K, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63);
    w.load_tables(threadIdx.x);
    __syncthreads();
    T sum[PER + 1];  // coefficients threadIdx.x + 512 k of the sample, then its body
#pragma unroll
    for (int k = 0; k <= PER; k++) sum[k] = 0;
#pragma unroll 1
    for (int pass = 0; pass < (MUX ? 2 : 1); pass++) {
        // MUX: pass 0 = c + t - mu, pass 1 = -c + f - mu
        const uint32_t* a = MUX ? inc : in0;
        const uint32_t* b = MUX ? (pass == 0 ? in1 : in0) : in1;
        const uint32_t sa = static_cast<uint32_t>(MUX ? (pass == 0 ? 1 : -1) : ca);
        const uint32_t sb = static_cast<uint32_t>(MUX ? 1 : cb);
        const uint32_t off = MUX ? 0u - mu0 : offset;
        const PwMask mask{a, b, sa, sb};
        w.rotate(true, mask.body<P>(off), mu, mask);
        __syncthreads();
        const T* ca0 = reinterpret_cast<const T*>(w.buf(0, 0, 0));
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = threadIdx.x + S::NT * k;
            sum[k] += i == 0 ? ca0[0] : static_cast<T>(0 - ca0[N - i]);
        }
        sum[PER] += reinterpret_cast<const T*>(w.buf(0, 1, 0))[0];
        __syncthreads();
    }
    // key switch of the sum over all eight waves; the sample and the partial
    // sums lie in transform buffers
    T* const sample = reinterpret_cast<T*>(w.buf(0, 0, 1));
    uint32_t* const red = reinterpret_cast<uint32_t*>(w.buf(0, 0, 2));
    static_assert(sizeof(sm.buf[0]) * 2 >= 8 * (n0 + 1) * 4 && sizeof(sm.buf[0]) >= (N + 1) * sizeof(T),
                  "buffers");
#pragma unroll
    for (int k = 0; k < PER; k++) sample[threadIdx.x + S::NT * k] = sum[k];
    if (threadIdx.x == 0) sample[N] = sum[PER];
    __syncthreads();
    if constexpr (MUX)
        key_switch_waves<TFHEpp::lvl20param, false, 8>(out, sample, nullptr, mux_sign, 0,
                                                       mux_sign > 0 ? mu : 0 - mu, ksk, red, w.wave,
                                                       w.lane);
    else
        key_switch_waves<TFHEpp::lvl20param, false, 8>(out, sample, nullptr, 1, 0, 0, ksk, red, w.wave,
                                                       w.lane);
}

// ---------------------------------------------------------------------------
// Batched key switching (gather form): one job per workgroup of eight waves,
// each wave taking 1/8 of the input coefficients for all output columns,
// partial sums reduced through LDS. One job's key switch is a long dependent
// gather loop (1024 x 7 KSK rows at lvl1, 2048 x 7 at lvl2), so a job on a
// single wave is latency-bound for milliseconds; split eight ways it is not.
template <class KS, bool SUBSET>
__global__ __launch_bounds__(512) void k_ks_batch(const KsJob* __restrict__ jobs, int njobs,
                                                  const uint32_t* ksk)
{
    using DT = typename KS::domainP::T;
    __shared__ uint32_t sh_red[8 * (KsTraits<KS>::n0 + 1)];
    const int job = blockIdx.x;
    if (job >= njobs) return;
    const KsJob jb = jobs[job];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    key_switch_waves<KS, SUBSET, 8>(jb.out, static_cast<const DT*>(jb.in0),
                                    static_cast<const DT*>(jb.in1), jb.ca, jb.cb,
                                    static_cast<DT>(jb.offset), ksk, sh_red, wave,
                                    threadIdx.x & 63);
}

// Elementwise TLWE combinations (MUX/NMUX combine, NOT, COPY).
__global__ __launch_bounds__(256) void k_linear(const LinJob* __restrict__ jobs, int njobs)
{
    const LinJob jb = jobs[blockIdx.x];
    for (int i = threadIdx.x; i < jb.words; i += 256) {
        uint32_t v = static_cast<uint32_t>(jb.s1) * jb.r1[i];
        if (jb.r0) v += static_cast<uint32_t>(jb.s0) * jb.r0[i];
        if (i == jb.words - 1) v += jb.offset;
        jb.out[i] = v;
    }
}

// One CMUX accumulate step on a TRLWE in global memory (reference
// include/gatebootstrapping_gpu.cuh:69-221): acc += ExtProd((X^a-1) acc, C).
template <class P>
__global__ __launch_bounds__(128, 2) void k_cmux_fft(typename P::T* trlwe, const cplx* trgsw,
                                                   uint32_t abar, FourierKeys<P> K)
{
    using T = typename P::T;
    constexpr int N = P::n, H = N / 2, R = N / 128;
    constexpr bool kL = AccStore<P>::kLds;
    constexpr int NB = BrShape<P>::NB;
    __shared__ cplx sh_spec[2][NB * H];
    __shared__ T sh_coef[kL ? 2 : 1][kL ? N : 1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    AccStore<P> acc;
    if constexpr (kL) acc.lds = sh_coef[wave];
#pragma unroll
    for (int r = 0; r < 2 * R; r++)
        acc.set(r, lane, trlwe[wave * N + AccStore<P>::coef_index(r, lane)]);
    if constexpr (kL) wave_lds_sync();
    br_step_fft<P, false>(acc, wave, abar, 0, trgsw, sh_spec[wave], sh_spec[wave ^ 1], K);
#pragma unroll
    for (int r = 0; r < 2 * R; r++)
        trlwe[wave * N + AccStore<P>::coef_index(r, lane)] = acc.get(r, lane);
}

// Batched lvl1 CMUX (reference src/bootstrap_gpu.cu:700-813 __CMUXNTT__,
// FFT build): res = c0 + ExtProd(c1 - c0, C), one workgroup of two waves per
// CMUX (wave j owns component j; the pair exchanges digit spectra through
// LDS). Each wave reads its own component of c1 and c0 before the first
// barrier and writes its component of res last, so res may alias c0 or c1.
template <class P>
__global__ __launch_bounds__(128, 2) void k_cmux_batch_fft(CmuxBatch batch, FourierKeys<P> K)
{
    static_assert(!AccStore<P>::kLds, "register accumulator (lvl1)");
    constexpr int N = P::n, R = N / 128;
    constexpr int NB = BrShape<P>::NB;
    __shared__ cplx sh_spec[2][NB * (N / 2)];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const CmuxDesc d = batch.at(blockIdx.x);
    AccStore<P> acc;
#pragma unroll
    for (int r = 0; r < 2 * R; r++) {
        const int i = wave * N + AccStore<P>::coef_index(r, lane);
        acc.set(r, lane, d.c1[i] - d.c0[i]);
    }
    br_step_fft<P, false, false, true>(acc, wave, 0, 0, static_cast<const cplx*>(d.cs),
                                       sh_spec[wave], sh_spec[wave ^ 1], K);
#pragma unroll
    for (int r = 0; r < 2 * R; r++) {
        const int i = wave * N + AccStore<P>::coef_index(r, lane);
        d.res[i] = d.c0[i] + acc.get(r, lane);
    }
}

// ---------------------------------------------------------------------------
// Launchers

void launch_cmux_batch_fft(const CmuxBatch& batch, int n, const FourierKeys<lvl1param>& K,
                           hipStream_t st)
{
    hipLaunchKernelGGL((k_cmux_batch_fft<lvl1param>), dim3(n), dim3(128), 0, st, batch, K);
}

template <class P>
void launch_to_fourier(cplx* out, const void* in, int npolys, bool integer,
                       const FourierKeys<P>& K, hipStream_t st)
{
    const dim3 grid((npolys + 3) / 4), block(256);
    if (integer)
        hipLaunchKernelGGL((k_to_fourier<P, true>), grid, block, 0, st, out, in, npolys, K);
    else
        hipLaunchKernelGGL((k_to_fourier<P, false>), grid, block, 0, st, out, in, npolys, K);
}
template void launch_to_fourier<lvl1param>(cplx*, const void*, int, bool,
                                           const FourierKeys<lvl1param>&, hipStream_t);
template void launch_to_fourier<lvl2param>(cplx*, const void*, int, bool,
                                           const FourierKeys<lvl2param>&, hipStream_t);

template <class P>
void launch_from_fourier(double* out, const cplx* in, int npolys, const FourierKeys<P>& K,
                         hipStream_t st)
{
    hipLaunchKernelGGL((k_from_fourier<P>), dim3((npolys + 3) / 4), dim3(256), 0, st, out, in,
                       npolys, K);
}
template void launch_from_fourier<lvl1param>(double*, const cplx*, int,
                                             const FourierKeys<lvl1param>&, hipStream_t);
template void launch_from_fourier<lvl2param>(double*, const cplx*, int,
                                             const FourierKeys<lvl2param>&, hipStream_t);

template <class P>
void launch_xai_poly(int32_t* out, hipStream_t st)
{
    hipLaunchKernelGGL((k_xai_poly<P>), dim3(2 * P::n), dim3(256), 0, st, out);
}
template void launch_xai_poly<lvl1param>(int32_t*, hipStream_t);
template void launch_xai_poly<lvl2param>(int32_t*, hipStream_t);

// lvl1 rotation (br_fft_pw.hpp) in the workgroups that fft_split gives.
template <bool KB, int J, int DPW, int PF, int HELP>
static void launch_pw_lvl1(const BrJob* jobs, int njobs, uint32_t mu,
                           const FourierKeys<lvl1param>& K, hipStream_t st)
{
    using S = PwShape<lvl1param, J, DPW, PF, HELP, KB>;
    if (njobs > 0)
        hipLaunchKernelGGL((k_br_fft_pw<S, 2>), dim3((njobs + J - 1) / J), dim3(S::NT), 0, st, jobs,
                           njobs, mu, K);
}
template <bool KB>
static void launch_br_lvl1(const BrJob* jobs, int njobs, int c, uint32_t mu,
                           const FourierKeys<lvl1param>& K, hipStream_t st)
{
    const FftSplit w = fft_split(KB, njobs, c, device_cu_count());
    if constexpr (KB)
        launch_pw_lvl1<true, 4, 2, 4, 0>(jobs, w.wide, mu, K, st);
    else
        launch_pw_lvl1<false, 2, 1, 8, 0>(jobs, w.wide, mu, K, st);
    if (w.width == 2)
        launch_pw_lvl1<KB, 2, 1, 8, 0>(jobs + w.wide, w.rest, mu, K, st);
    else
        launch_pw_lvl1<KB, 1, 1, 8, 4>(jobs + w.wide, w.rest, mu, K, st);
}

// lvl2 rotation. Key bundle (c = 1): br_fft_pw.hpp, one job per workgroup and
// CU; CMUX keys, or c = 2 (a tuning option, two jobs per workgroup): two waves
// per job. All in a resident grid with a grid stride: the key (167 MB, bundle
// 250 MB) outgrows the caches once the workgroups drift apart.
// The bundle's workgroup fills a CU's LDS, so batches of several streams share
// no CU as the two-wave workgroups did, two to a CU. Plans of 1 to 900 gates on
// two to eight streams are up to 2.2 times as fast all the same, but where all of
// them together are up to a sixth over a job per CU: the few left then rotate in
// a round of their own, with the key from memory (two streams of 130 gates 10.7
// ms, of 150 10.0, of 200 9.5; 9.8 before).
template <bool KB, int C>
static void launch_br_two_wave(const BrJob* jobs, int njobs, uint64_t mu,
                               const FourierKeys<lvl2param>& K, hipStream_t st)
{
    const int groups = (njobs + C - 1) / C, cap = br_fft_resident_groups<KB, C>();
    hipLaunchKernelGGL((k_br_fft<KB, C>), dim3(cap > 0 && groups > cap ? cap : groups),
                       dim3(128 * C), 0, st, jobs, njobs, mu, K);
}
template <bool KB>
static void launch_br_lvl2(const BrJob* jobs, int njobs, int c, uint64_t mu,
                           const FourierKeys<lvl2param>& K, hipStream_t st)
{
    const int cus = device_cu_count();
    if (c == 2)
        launch_br_two_wave<KB, 2>(jobs, njobs, mu, K, st);
    else if constexpr (KB)
        hipLaunchKernelGGL((k_br_fft_pw<Lvl2Shape, 2>), dim3(njobs < cus ? njobs : cus),
                           dim3(Lvl2Shape::NT), 0, st, jobs, njobs, mu, K);
    else
        launch_br_two_wave<KB, 1>(jobs, njobs, mu, K, st);
}

template <class P, bool KB>
void launch_br_fft(const BrJob* jobs, int njobs, int c, typename P::T mu,
                   const FourierKeys<P>& K, hipStream_t st)
{
    if (njobs <= 0) return;
    if constexpr (sizeof(typename P::T) == 4)
        launch_br_lvl1<KB>(jobs, njobs, c, mu, K, st);
    else
        launch_br_lvl2<KB>(jobs, njobs, c, mu, K, st);
}
template void launch_br_fft<lvl1param, true>(const BrJob*, int, int, uint32_t,
                                             const FourierKeys<lvl1param>&, hipStream_t);
template void launch_br_fft<lvl1param, false>(const BrJob*, int, int, uint32_t,
                                              const FourierKeys<lvl1param>&, hipStream_t);
template void launch_br_fft<lvl2param, true>(const BrJob*, int, int, uint64_t,
                                             const FourierKeys<lvl2param>&, hipStream_t);
template void launch_br_fft<lvl2param, false>(const BrJob*, int, int, uint64_t,
                                              const FourierKeys<lvl2param>&, hipStream_t);

void launch_gate_lvl1_fft(bool kb, bool mux, uint32_t* out, const uint32_t* in0,
                          const uint32_t* in1, const uint32_t* inc, int32_t ca, int32_t cb,
                          uint32_t offset, int32_t mux_sign, const uint32_t* ksk,
                          const FourierKeys<lvl1param>& K, hipStream_t st)
{
#define CUFHE_L(KBV, MUXV)                                                                     \
    hipLaunchKernelGGL((k_gate_lvl1_pw<KBV, MUXV>), dim3(1), dim3(512), 0, st, out, in0, in1, inc, \
                       ca, cb, offset, mux_sign, ksk, K)
    if (kb) {
        if (mux) CUFHE_L(true, true); else CUFHE_L(true, false);
    }
    else {
        if (mux) CUFHE_L(false, true); else CUFHE_L(false, false);
    }
#undef CUFHE_L
}

void launch_gate_lvl01_fft(bool kb, bool mux, bool subset, uint32_t* out, const uint32_t* in0,
                           const uint32_t* in1, const uint32_t* inc, int32_t ca, int32_t cb,
                           uint32_t offset, int32_t mux_sign, uint32_t tv_mu, const uint32_t* ksk,
                           const FourierKeys<lvl1param>& K, hipStream_t st)
{
#define CUFHE_G01(KBV, MUXV, SUB)                                                                 \
    hipLaunchKernelGGL((k_gate_lvl01_pw<KBV, MUXV, SUB>), dim3(1), dim3(512), 0, st, out, in0, in1, \
                       inc, ca, cb, offset, mux_sign, tv_mu, ksk, K)
#define CUFHE_G01S(KBV, MUXV)                                                      \
    do {                                                                           \
        if (subset) CUFHE_G01(KBV, MUXV, true); else CUFHE_G01(KBV, MUXV, false); \
    } while (0)
    if (kb) {
        if (mux) CUFHE_G01S(true, true); else CUFHE_G01S(true, false);
    }
    else {
        if (mux) CUFHE_G01S(false, true); else CUFHE_G01S(false, false);
    }
#undef CUFHE_G01S
#undef CUFHE_G01
}

void launch_se_ks_lvl10(bool subset, uint32_t* out, const uint32_t* trlwe, int n,
                        const uint32_t* ksk, hipStream_t st)
{
    if (n <= 0) return;
    if (subset)
        hipLaunchKernelGGL((k_se_ks_lvl10<true>), dim3(n), dim3(512), 0, st, out, trlwe, n, ksk);
    else
        hipLaunchKernelGGL((k_se_ks_lvl10<false>), dim3(n), dim3(512), 0, st, out, trlwe, n, ksk);
}

void launch_gate_lvl02_fft(bool kb, bool mux, uint32_t* out, const uint32_t* in0,
                           const uint32_t* in1, const uint32_t* inc, int32_t ca, int32_t cb,
                           uint32_t offset, int32_t mux_sign, const uint32_t* ksk,
                           const FourierKeys<lvl2param>& K, hipStream_t st)
{
    const dim3 grid(1);
#define CUFHE_L(MUXV)                                                                          \
    hipLaunchKernelGGL((k_gate_lvl02_fft<MUXV>), grid, dim3(256), 0, st, out, in0, in1, inc, ca, \
                       cb, offset, mux_sign, ksk, K)
    if (kb) {
        if (mux)
            hipLaunchKernelGGL((k_gate_lvl02_pw<true>), grid, dim3(512), 0, st, out, in0, in1, inc, ca,
                               cb, offset, mux_sign, ksk, K);
        else
            hipLaunchKernelGGL((k_gate_lvl02_pw<false>), grid, dim3(512), 0, st, out, in0, in1, inc, ca,
                               cb, offset, mux_sign, ksk, K);
    }
    else {
        if (mux) CUFHE_L(true); else CUFHE_L(false);
    }
#undef CUFHE_L
}

void launch_ks_batch(int domain_level, bool subset, const KsJob* jobs, int njobs,
                     const uint32_t* ksk, hipStream_t st)
{
    if (njobs <= 0) return;
    const dim3 grid(njobs), block(512);
    if (domain_level == 1) {
        if (subset)
            hipLaunchKernelGGL((k_ks_batch<TFHEpp::lvl10param, true>), grid, block, 0, st, jobs,
                               njobs, ksk);
        else
            hipLaunchKernelGGL((k_ks_batch<TFHEpp::lvl10param, false>), grid, block, 0, st,
                               jobs, njobs, ksk);
    }
    else {
        hipLaunchKernelGGL((k_ks_batch<TFHEpp::lvl20param, false>), grid, block, 0, st, jobs,
                           njobs, ksk);
    }
}

__global__ __launch_bounds__(256) void k_linear_one(LinJob jb)
{
    for (int i = threadIdx.x; i < jb.words; i += 256) {
        uint32_t v = static_cast<uint32_t>(jb.s1) * jb.r1[i];
        if (jb.r0) v += static_cast<uint32_t>(jb.s0) * jb.r0[i];
        if (i == jb.words - 1) v += jb.offset;
        jb.out[i] = v;
    }
}

void launch_linear_one(const LinJob& jb, hipStream_t st)
{
    hipLaunchKernelGGL(k_linear_one, dim3(1), dim3(256), 0, st, jb);
}

void launch_linear(const LinJob* jobs, int njobs, hipStream_t st)
{
    hipLaunchKernelGGL(k_linear, dim3(njobs), dim3(256), 0, st, jobs, njobs);
}

template <class P>
void launch_cmux_fft(typename P::T* trlwe, const cplx* trgsw, uint32_t abar,
                     const FourierKeys<P>& K, hipStream_t st)
{
    hipLaunchKernelGGL((k_cmux_fft<P>), dim3(1), dim3(128), 0, st, trlwe, trgsw, abar, K);
}
template void launch_cmux_fft<lvl1param>(uint32_t*, const cplx*, uint32_t,
                                         const FourierKeys<lvl1param>&, hipStream_t);
template void launch_cmux_fft<lvl2param>(uint64_t*, const cplx*, uint32_t,
                                         const FourierKeys<lvl2param>&, hipStream_t);

}  // namespace cufhe_amd
