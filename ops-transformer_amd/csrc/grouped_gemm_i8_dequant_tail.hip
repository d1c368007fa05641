// Expert-grouped int8 GEMM: the LDS-ring kernels of the kDequant epilogue for K off the 128 grid (see kTail in
// grouped_gemm_i8_kernels.h).
#include "grouped_gemm_i8_kernels.h"

namespace gemm {

hipError_t LaunchRingTailDequant(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream) {
    return LaunchStreamShape<Epilogue::kDequant, true>(plan, args, sched, stream);
}

}  // namespace gemm
