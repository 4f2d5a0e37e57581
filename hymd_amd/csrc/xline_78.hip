// x-line pass (xline.h) for 7 and 8 types.
#include "xline.h"

namespace hymd {

int xline_pass_7(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<7, false, 3, 4, 5>(plan, sh, job, blocks, s);
}

int xline_pass_8(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<8, false, 3, 4, 5>(plan, sh, job, blocks, s);
}

}  // namespace hymd
