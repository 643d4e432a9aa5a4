// How far the lvl1 key-bundle product lies from the integers that its exact value
// is, before the rounding to Torus32: the rotation's transforms (fft512.hpp, with
// X^(a0+a1) as the product of two roots) and the radix-8 transforms of
// fft_wave.hpp (with X^(a0+a1) from the table), lane by lane on the host,
// against integer convolutions. Runs without a GPU.
#include "../../cufhe_amd/csrc/device_common.hpp"
#include "../../cufhe_amd/csrc/fft_tables.hpp"

#include <algorithm>
#include <cstdio>
#include <cstdlib>

using namespace cufhe_amd;

constexpr int N = 1024, H = 512, L = 2, ROWS = 4;
using Lanes = cplx[64][8];

static const FoldedTables tabs(N);
static const FFTTables radix8{tabs.twl.data(), tabs.tw64.data(), tabs.cr.data(), tabs.tws.data()};
static const std::vector<cplx> roots = fft512_tables();

static uint64_t rnd_state = 88172645463325252ull;
static uint64_t rnd()
{
    rnd_state ^= rnd_state << 13;
    rnd_state ^= rnd_state >> 7;
    rnd_state ^= rnd_state << 17;
    return rnd_state;
}

template <class F>
static void each_lane(F&& f)
{
    for (int lane = 0; lane < 64; lane++) f(lane);
}

// forward transform of p (times scale); spec[512] in storage order
static void forward_radix8(const int64_t* p, double scale, cplx* spec)
{
    using namespace fft_stage;
    static Lanes x;
    static cplx buf[kScratchPad(H)];
    each_lane([&](int l) {
        for (int r = 0; r < 8; r++) x[l][r] = cplx{p[l + 64 * r] * scale, p[l + 64 * r + H] * scale};
        fwd_a<8>(x[l], radix8, l);
        t1_store<8>(x[l], buf, l);
    });
    each_lane([&](int l) { t1_load<8>(x[l], buf, l); });
    each_lane([&](int l) {
        fwd_b<8>(x[l], radix8, l);
        t2_store_cx<8>(x[l], buf, l);
    });
    each_lane([&](int l) {
        t2_load_xc<8>(x[l], buf, l);
        fwd_c<8>(x[l]);
        for (int d = 0; d < 8; d++) spec[d * 64 + l] = x[l][d];
    });
}
// inverse, in Torus32 units
static void inverse_radix8(const cplx* spec, double* v)
{
    using namespace fft_stage;
    static Lanes x;
    static cplx buf[kScratchPad(H)];
    each_lane([&](int l) {
        for (int d = 0; d < 8; d++) x[l][d] = spec[d * 64 + l];
        inv_a<8>(x[l]);
        t2_store_xc<8>(x[l], buf, l);
    });
    each_lane([&](int l) { t2_load_cx<8>(x[l], buf, l); });
    each_lane([&](int l) {
        inv_b<8>(x[l], radix8, l);
        t1_store_inv<8>(x[l], buf, l);
    });
    each_lane([&](int l) {
        t1_load_inv<8>(x[l], buf, l);
        inv_c<8>(x[l], radix8, l);
        for (int r = 0; r < 8; r++) {
            v[l + 64 * r] = x[l][r].x * (4294967296.0 / H);
            v[l + 64 * r + H] = x[l][r].y * (4294967296.0 / H);
        }
    });
}

// the same by fft512.hpp's stages
static void forward_512(const int64_t* p, cplx* spec)
{
    using namespace fft512;
    static Lanes x;
    static cplx buf[kScratch];
    each_lane([&](int l) {
        for (int r = 0; r < 8; r++)
            x[l][r] = cplx{static_cast<double>(p[l + 64 * r]), static_cast<double>(p[l + 64 * r + H])};
        levels(x[l], first_roots());
        for (int r = 0; r < 8; r++) buf[row1(r) + l] = x[l][r];
    });
    each_lane([&](int l) {
        for (int b = 0; b < 8; b++) x[l][b] = buf[octet_row1(l) + 8 * b];
    });
    each_lane([&](int l) {
        levels(x[l], load_roots<8>(roots.data(), l >> 3));
        for (int c = 0; c < 8; c++) buf[sub_a(l) + 9 * c] = x[l][c];
    });
    each_lane([&](int l) {
        for (int a = 0; a < 8; a++) x[l][a] = buf[sub_b(l) + a];
        levels(x[l], load_roots<64>(roots.data() + kTab1, l));
        const Slots s = Slots::of(l);
        for (int a = 0; a < 8; a++) spec[s.at(a)] = x[l][a];
    });
}
// inverse, in turns
static void inverse_512(const cplx* spec, double* v)
{
    using namespace fft512;
    static Lanes x;
    static cplx buf[kScratch];
    each_lane([&](int l) {
        const Slots s = Slots::of(l);
        for (int a = 0; a < 8; a++) x[l][a] = spec[s.at(a)];
        const Roots r = load_roots<64>(roots.data() + kTab1, l);
        ilevels(x[l], r);
        rescale(x[l], r);
        for (int a = 0; a < 8; a++) buf[sub_b(l) + a] = x[l][a];
    });
    each_lane([&](int l) {
        for (int c = 0; c < 8; c++) x[l][c] = buf[sub_a(l) + 9 * c];
    });
    each_lane([&](int l) {
        const Roots r = load_roots<8>(roots.data(), l >> 3);
        ilevels(x[l], r);
        rescale(x[l], r);
        for (int b = 0; b < 8; b++) buf[octet_row1(l) + 8 * b] = x[l][b];
    });
    each_lane([&](int l) {
        for (int r = 0; r < 8; r++) x[l][r] = buf[row1(r) + l];
        ilevels(x[l], first_roots());
        for (int r = 0; r < 8; r++) {
            const double s = scale(first_roots(), r) / H;
            v[l + 64 * r] = x[l][r].x * s;
            v[l + 64 * r + H] = x[l][r].y * s;
        }
    });
}

// X^a at storage place d * 64 + lane
static cplx root_at(uint32_t a, int d, int lane)
{
    const int kb = (lane >> 3) + 8 * (lane & 7);
    const int m = static_cast<int>((a * static_cast<uint32_t>(d)) & 7u) * 2;
    return cmul(tabs.e2n[static_cast<int>(a) * (1 - 4 * kb) & (2 * N - 1)], cplx{cos16(m), -sin16(m)});
}

static void mul_x_minus_1(const int64_t* p, uint32_t a, int64_t* out)  // out += (X^a - 1) p
{
    for (int i = 0; i < N; i++) {
        const uint32_t t = (i + a) & (2 * N - 1);
        out[t & (N - 1)] += t < N ? p[i] : -p[i];
        out[i] -= p[i];
    }
}

struct Error {
    double max = 0, sum = 0;
    long n = 0, wrong = 0;
    void add(double e)
    {
        max = std::max(max, std::fabs(e));
        sum += e * e;
        n++;
    }
    double rms() const { return std::sqrt(sum / n); }
};

// One product: digits[row][N], one output column, key[member][row][N] as signed
// words, members (both, first, second) of exponents a0 + a1, a0, a1.
static void product(const int64_t (*digits)[N], const int64_t (*key)[ROWS][N], int col, uint32_t a0, uint32_t a1,
                    Error& six, Error& eight)
{
    static int64_t want[N];
    static cplx k[3][ROWS][H], d[H];
    static cplx s6[H], s8[H];
    std::fill(want, want + N, 0);
    for (int i = 0; i < H; i++) s6[i] = s8[i] = cplx{0, 0};
    for (int row = 0; row < ROWS; row++) {
        const int q = row % L;
        static int64_t b[N];
        std::fill(b, b + N, 0);
        mul_x_minus_1(key[0][row], a0 + a1, b);
        mul_x_minus_1(key[1][row], a0, b);
        mul_x_minus_1(key[2][row], a1, b);
        if (row / L == col) b[0] += 1ll << (32 - 8 * (q + 1));
        for (int i = 0; i < N; i++) {
            const int64_t v = digits[row][i];
            for (int j = 0; j < N - i; j++) want[i + j] += v * b[j];
            for (int j = N - i; j < N; j++) want[i + j - N] -= v * b[j];
        }
        for (int e = 0; e < 3; e++) forward_radix8(key[e][row], 1.0 / 4294967296.0, k[e][row]);
        const double hq = row / L == col ? std::ldexp(1.0, -8 * (q + 1)) : 0.0;
        for (int form = 0; form < 2; form++) {
            if (form)
                forward_radix8(digits[row], 1.0, d);
            else
                forward_512(digits[row], d);
            for (int p = 0; p < H; p++) {
                cplx x0 = root_at(a0, p >> 6, p & 63), x1 = root_at(a1, p >> 6, p & 63);
                cplx x01 = form ? root_at(a0 + a1, p >> 6, p & 63) : cmul(x0, x1);
                x0.x -= 1.0;
                x1.x -= 1.0;
                x01.x -= 1.0;
                cplx t{hq, 0.0};
                cmac(t, k[2][row][p], x1);
                cmac(t, k[1][row][p], x0);
                cmac(t, k[0][row][p], x01);
                cmac((form ? s8 : s6)[p], d[p], t);
            }
        }
    }
    static double v[N];
    inverse_512(s6, v);
    for (int i = 0; i < N; i++) {
        six.add(static_cast<double>(static_cast<long double>(v[i]) * 4294967296.0L - want[i]));
        if (turns_to_torus32(v[i]) != static_cast<uint32_t>(want[i])) six.wrong++;
    }
    inverse_radix8(s8, v);
    for (int i = 0; i < N; i++) eight.add(static_cast<double>(static_cast<long double>(v[i]) - want[i]));
}

int main()
{
    static int64_t digits[ROWS][N], key[3][ROWS][N];
    Error six, eight;
    for (int trial = 0; trial < 60; trial++) {
        for (auto& row : digits)
            for (auto& v : row) v = static_cast<int64_t>(rnd() % 256) - 128;
        for (auto& e : key)
            for (auto& row : e)
                for (auto& v : row) v = static_cast<int32_t>(rnd() >> 32);
        product(digits, key, trial & 1, rnd() % (2 * N), rnd() % (2 * N), six, eight);
    }
    std::printf("distance from the integer, units of 2^-32: six-FMA transforms rms %.3g max %.3g, radix-8 rms %.3g "
                "max %.3g\n",
                six.rms(), six.max, eight.rms(), eight.max);
    // a coefficient's terms are independent, so its error is near normal: 1/8 unit,
    // a quarter of the way to another word, is 14 times the rms
    if (six.wrong || six.max > 0.125 || six.rms() > eight.rms()) return 1;
    std::printf("ok: %ld coefficients\n", six.n);
    return 0;
}
