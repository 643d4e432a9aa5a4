// The launch rules of the lvl1 rotations on the host, for every batch size up to
// twelve thousand and several CU counts. Runs without a GPU.
#include "../../cufhe_amd/csrc/launch_rules.hpp"

#include <cstdio>
#include <cstdlib>

using namespace cufhe_amd;

static long checked = 0;
static void require(bool ok, const char* what, int njobs, int cus)
{
    if (!ok) {
        std::printf("%s: %d jobs on %d CUs\n", what, njobs, cus);
        std::exit(1);
    }
    checked++;
}
static int ceil_div(int a, int b) { return (a + b - 1) / b; }

// every workgroup has 1 .. 8 jobs, in as few rounds of workgroups as eight jobs take
static void check_ntt(bool cmux, int njobs, int cus)
{
    const int groups = ntt_workgroups(cmux, njobs, cus);
    require(groups >= 1 && groups <= njobs, "empty workgroups", njobs, cus);
    require(ceil_div(njobs, groups) <= kNttPwJobs, "more than eight jobs", njobs, cus);
    require(ceil_div(groups, cus) == ceil_div(njobs, kNttPwJobs * cus), "rounds", njobs, cus);
    // CMUX keys: a batch of up to two jobs a CU leaves half of the CUs free
    if (cmux && njobs <= 2 * cus && cus > 1)
        require(groups <= std::max(cus / 2, ceil_div(njobs, 2)), "whole card", njobs, cus);
}

// the jobs are covered, full workgroups first; the default takes no more rounds of
// workgroups than a fixed width, and c = 6 is the default
static void check_fft(bool bundle, int njobs, int cus)
{
    const FftSplit d = fft_split(bundle, njobs, 8, cus);
    auto groups = [](const FftSplit& s) { return ceil_div(s.wide, s.most) + ceil_div(s.rest, s.width); };
    for (int c : {1, 2, 4, 6, 8}) {
        const FftSplit s = fft_split(bundle, njobs, c, cus);
        require(s.wide >= 0 && s.rest >= 0 && s.wide + s.rest == njobs, "coverage", njobs, cus);
        require(s.most == (bundle ? 4 : 2) && (s.width == 1 || s.width == 2), "widths", njobs, cus);
        require(ceil_div(groups(d), cus) <= ceil_div(groups(s), cus), "rounds", njobs, cus);
    }
    require(d == fft_split(bundle, njobs, 6, cus), "c = 6", njobs, cus);
    require((d == fft_split(bundle, njobs, 4, cus)) || (bundle && d.rest > 0), "c = 4", njobs, cus);
    // a fixed width that does the same as the default is the same launch
    if (njobs <= cus) require(d == fft_split(bundle, njobs, 1, cus), "c = 1", njobs, cus);
    if (njobs == 2 * cus) require(d == fft_split(bundle, njobs, 2, cus), "c = 2", njobs, cus);
}

// the default stays unless every repeat of another launch was faster
static void check_tuned_choice()
{
    const TunedTime noise[] = {{8, 10.88f, 10.95f}, {4, 10.86f, 10.90f}, {2, 14.f, 14.1f}};
    require(tuned_choice(noise, 3) == 8, "a tie", 0, 0);
    const TunedTime faster[] = {{8, 10.8f, 10.9f}, {4, 9.9f, 10.7f}, {2, 9.5f, 9.6f}, {1, 9.0f, 10.9f}};
    require(tuned_choice(faster, 4) == 2, "a faster launch", 0, 0);
    require(tuned_choice(faster, 1) == 8, "one launch", 0, 0);
}

int main()
{
    check_tuned_choice();
    for (int cus : {1, 32, 80, 256, 304})
        for (int njobs = 1; njobs <= 12000; njobs++)
            for (bool cmux : {false, true}) {
                check_ntt(cmux, njobs, cus);
                check_fft(!cmux, njobs, cus);
            }
    std::printf("ok: %ld checks\n", checked);
    return 0;
}
