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

// Workgroups of an lvl1 FFT batch (br_fft_pw.hpp): its first `wide` jobs in
// workgroups of `most`, the rest in workgroups of `width`. Key bundle, c = 1, 2, 4:
// that many jobs per workgroup throughout; else (6, 8, the default) the mix that
// takes the fewest rounds of the CUs: four jobs per CU share a key pass and the LDS
// best (2.97 ms a round of 1024 jobs, 11.3 ms for 4096), a CU with two or one is
// done sooner (1.78 ms for 512, 1.21 ms for 256; MI355X). So full rounds run
// at four and what is left at the smallest width that holds it in one round.
// Eight-wave workgroups of one wave per job, the form before, took 3.5 / 3.7 /
// 4.2 / 12.0 ms for 256 / 512 / 1024 / 4096 jobs.
// CMUX keys (one TRGSW per key bit) add the accumulators to the LDS, so two
// jobs per workgroup are the most; c = 4 and 8 (the default) mix two and one.
struct FftSplit {
    int most, wide, rest, width;
    bool operator==(const FftSplit& o) const
    {
        return most == o.most && wide == o.wide && rest == o.rest && width == o.width;
    }
    int workgroups() const { return (wide + most - 1) / most + (rest + width - 1) / width; }
};
inline FftSplit fft_split(bool bundle, int njobs, int c, int cus)
{
    const int most = bundle ? 4 : 2;
    int wide = 0;
    if (c == most) {
        wide = njobs;
    }
    else if (c != 1 && c != 2) {
        wide = njobs / (most * cus) * (most * cus);
        if (njobs - wide > most / 2 * cus) wide = njobs;
    }
    const int rest = njobs - wide;
    return FftSplit{most, wide, rest, rest > 0 && (c == 2 || (c != 1 && rest > cus)) ? 2 : 1};
}

// Times of one launch of a batch over a few repeats.
struct TunedTime {
    int c;
    float best, worst;
};
// The c of the fastest of n launches, where the first is the default: another one is
// taken only if every repeat of it was faster than the default's best, because the
// pick goes on to smaller batches, where a fixed width can take more than twice the
// default's time (150 jobs at four a workgroup 2.97 ms, the default 1.21).
inline int tuned_choice(const TunedTime* t, int n)
{
    int pick = 0;
    for (int i = 1; i < n; i++)
        if (t[i].worst < t[0].best && t[i].best < t[pick].best) pick = i;
    return t[pick].c;
}

}  // namespace cufhe_amd
