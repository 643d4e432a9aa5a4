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

int main()
{
    for (int cus : {1, 32, 80, 256, 304})
        for (int njobs = 1; njobs <= 12000; njobs++)
            for (bool cmux : {false, true}) check_ntt(cmux, njobs, cus);
    std::printf("ok: %ld checks\n", checked);
    return 0;
}
