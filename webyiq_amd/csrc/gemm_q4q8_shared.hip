// The prefill GEMM's 128-token tiles with two workgroups per CU (gemm_q4q8.hip
// describes the kernel and its plan): the instances with one wave group.
#include "gemm_tile.hpp"

namespace wq {

hipError_t launch_gemm_shared(const LinearArgs& a, int bn, hipStream_t s) {
    if (a.acc_dump) {  // a test hook: the group sums of the same instances
        switch (bn) {
            case 192: return launch_tile<192, 1, true>(a, s);
            case 128: return launch_tile<128, 1, true>(a, s);
            default: return launch_tile<64, 1, true>(a, s);
        }
    }
    switch (bn) {
        case 192: return launch_tile<192, 1, false>(a, s);
        case 128: return launch_tile<128, 1, false>(a, s);
        default: return launch_tile<64, 1, false>(a, s);
    }
}

}  // namespace wq
