// x-line pass (xline.h): shapes and dispatch, and the one- and two-type kernels.
#include <algorithm>

#include "xline.h"

namespace hymd {

// Lines per workgroup.  A line needs n / R2 threads (one per last-stage
// butterfly); wider workgroups read longer runs of an x row (8 W bytes) and
// narrower ones give the chip more blocks, so: 16 lines, halved while they
// exceed the threads, half of a CU's LDS or a middle stage's registers, or
// while the blocks would not fill the chip twice and the runs are longer than
// 32 bytes.  Eight types fill a block's threads by themselves, so there once
// is enough (update of 64^3, 264 blocks of 8 lines 98 us, 528 of 4 103; seven
// types 92 and 88).
XlineShape xline_shape(const FftPlan &plan, int T, int want, bool fixed) {
    XlineShape sh;
    const int n = plan.mesh.mx, lines = plan.mesh.my * plan.mesh.zh;
    if (T < 1 || T > 8) return sh;
    const int fixed_lines = fixed ? xline_fixed_lines(n, T, want) : 0;
    sh.plan = xline_plan_of(T);
    const LineAxis &ax = plan.xl[sh.plan].fwd;
    if (ax.ns < 2) return sh;  // no fixed pass either
    const int nr2 = ax.st[ax.ns - 1].nr;
    auto threads = [&](int W) {
        const int t = std::max(W * nr2, std::min(256, T * W * ax.st[0].nr));
        return (t + 63) / 64 * 64;
    };
    auto fits = [&](int W, size_t lds) {
        if (threads(W) > kXlineThreads || xline_lds(n, T, W) > lds) return false;
        for (int s = 1; s < ax.ns - 1; ++s)  // the middle stages (the inverse plan's have the same radices)
            if (T * W * ax.st[s].nr > threads(W) * std::max(1, kXlineElems / ax.st[s].R)) return false;
        return true;
    };
    if (want > 0 && want != fixed_lines && fits(want, kXlineLdsBytes)) {
        sh.W = want;
    } else if (fixed_lines > 0) {
        sh.W = fixed_lines;
        sh.fixed = true;
        return sh;
    } else {
        for (int W = 16; W >= 8 && !sh.W; W >>= 1)
            if (threads(W) <= 256 && fits(W, 40 * 1024)) sh.W = W;
        for (int W = 16; W >= 2 && !sh.W; W >>= 1)
            if (fits(W, 80 * 1024)) sh.W = W;
        while (sh.W > 4 && lines / sh.W < (T < 8 ? 512 : 256) && fits(sh.W / 2, 80 * 1024)) sh.W /= 2;
        for (int W = 2; W >= 1 && !sh.W; W >>= 1)
            if (fits(W, kXlineLdsBytes)) sh.W = W;
    }
    sh.threads = sh.W ? threads(sh.W) : 0;
    // One line of one or two types (which keep the pass, xline_narrow): two or
    // four, where the middle stages need at most a quarter more threads for them
    // than the others.  900 x 96 x 96, one type 257 us with one line, 224 with
    // four; 900 x 256 x 256 2619 and 1574, its PME 2657 and 1632; 450 x 96 x 96, two
    // types 210 and 186.  (810 x 96 x 96, two types: half as many more, 366 and 382.)
    for (int W = 4; W >= 2 && T <= 2 && sh.W == 1; W >>= 1) {
        int t = threads(W);
        for (int s = 1; s < ax.ns - 1; ++s) {
            const int held = std::max(1, kXlineElems / ax.st[s].R);
            t = std::max(t, ((T * W * ax.st[s].nr + held - 1) / held + 63) / 64 * 64);
        }
        if (t > kXlineThreads || 4 * t > 5 * threads(W) || xline_lds(n, T, W) > 80 * 1024) continue;
        sh.W = W;
        sh.threads = t;
    }
    return sh;
}

int xline_pass(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int *nblocks, hipStream_t s) {
    static XlineLaunch *const by_types[8] = {xline_pass_1, xline_pass_2, xline_pass_3, xline_pass_4,
                                             xline_pass_5, xline_pass_6, xline_pass_7, xline_pass_8};
    HYMD_REQUIRE(sh.W > 0 && job.T >= 1 && job.T <= 8 && (!job.pme || job.T == 1), "no x-line pass for this job");
    const int blocks = (job.g.my * job.g.zh + sh.W - 1) / sh.W;
    *nblocks = blocks;
    if (sh.fixed) return xline_pass_fixed(plan, sh, job, blocks, s);
    return (job.pme ? xline_pass_pme : by_types[job.T - 1])(plan, sh, job, blocks, s);
}

int xline_pass_pme(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<1, true, 3, 4, 5, 6, 8, 10, 12, 15, 16>(plan, sh, job, blocks, s);
}

int xline_pass_1(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<1, false, 3, 4, 5, 6, 8, 10, 12, 15, 16>(plan, sh, job, blocks, s);
}

int xline_pass_2(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<2, false, 3, 4, 5, 6, 8, 10, 12, 15, 16>(plan, sh, job, blocks, s);
}

}  // namespace hymd
