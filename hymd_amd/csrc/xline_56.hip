// x-line pass (xline.h) for 5 and 6 types.
#include "xline.h"

namespace hymd {

int xline_pass_5(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<5, false, 3, 4, 5, 6>(plan, sh, job, blocks, s);
}

int xline_pass_6(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<6, false, 3, 4, 5>(plan, sh, job, blocks, s);
}

}  // namespace hymd
