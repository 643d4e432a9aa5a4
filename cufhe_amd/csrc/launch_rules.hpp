// The workgroups that a batch of lvl1 rotations is launched in, as plain
// functions of its size and the number of CUs.
#pragma once

#include <algorithm>

namespace cufhe_amd {

// Jobs that a workgroup of the NTT rotation (br_ntt_pw.hpp) has room for.
constexpr int kNttPwJobs = 8;

// Workgroups of an NTT batch; its jobs are spread evenly over them. A CU holds
// one workgroup, so a batch takes the fewest rounds of workgroups that hold it
// (block-binary rotations, 1, 2, 4 and 8 jobs a CU: 1.35, 1.55, 2.30 and 4.20 ms;
// 8 jobs in one round beat two rounds of 4, and 9 as 5 and 4 beat 8 and 1). No
// smaller width is offered: one job a workgroup in more rounds took 20.7 ms for
// 4096 block-binary jobs (fewest rounds 8.35) and 74.5 ms with CMUX keys (27.4).
// With CMUX keys a pair of jobs takes little longer than one (4.93 and 4.68 ms),
// so a batch that would take more than half of the CUs with a job each goes in
// pairs and leaves the others to batches of other streams: three streams of 256
// jobs 10.1 ms, with a job a CU 14.1. The other keys' pairs are dearer (1.55
// against 1.35 and 2.85 against 2.50 ms) and single jobs are kept.
inline int ntt_workgroups(bool cmux, int njobs, int cus)
{
    const int per_round = kNttPwJobs * cus;
    const int rounds = (njobs + per_round - 1) / per_round;
    if (cmux && 2 * njobs > cus && njobs <= 2 * cus) return (njobs + 1) / 2;
    return std::min(njobs, rounds * cus);
}

}  // namespace cufhe_amd
