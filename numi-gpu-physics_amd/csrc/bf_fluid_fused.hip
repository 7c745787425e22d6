// Instantiations of the fluid kernels with fused arithmetic for FP32
// populations and every collision operator (one unit per storage: they are
// the library's slowest to compile).
#include "bf_fluid.h"

namespace bf {

hipError_t launch_fluid_step_fused(int coll, const FluidBuffers& b, const StepParams& p, int parts, uint32_t wall_blocks,
                                  hipStream_t s) {
    switch (coll) {
        case COLL_TRT: return launch_step_t<ARITH_FUSED, COLL_TRT, STORE_FP32>(b, p, parts, wall_blocks, s);
        case COLL_TRT_SYMMETRIC_LIMITER:
            return launch_step_t<ARITH_FUSED, COLL_TRT_SYMMETRIC_LIMITER, STORE_FP32>(b, p, parts, wall_blocks, s);
        case COLL_REGULARIZED: return launch_step_t<ARITH_FUSED, COLL_REGULARIZED, STORE_FP32>(b, p, parts, wall_blocks, s);
        case COLL_RR3: return launch_step_t<ARITH_FUSED, COLL_RR3, STORE_FP32>(b, p, parts, wall_blocks, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace bf
