// x-line pass (xline.h) for 3 and 4 types.
#include "xline.h"

namespace hymd {

int xline_pass_3(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<3, false, 3, 4, 5, 6, 8>(plan, sh, job, blocks, s);
}

int xline_pass_4(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    return launch_xline_radix<4, false, 3, 4, 5, 6>(plan, sh, job, blocks, s);
}

}  // namespace hymd
