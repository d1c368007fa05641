// Expert-grouped int8 GEMM: the LDS-ring kernels of the kSwiglu epilogue for K off the 128 grid (see kTail in
// grouped_gemm_i8_kernels.h).
#include "grouped_gemm_i8_kernels.h"

namespace gemm {

hipError_t LaunchRingTailSwiglu(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream) {
    return LaunchStreamShape<Epilogue::kSwiglu, true>(plan, args, sched, stream);
}

}  // namespace gemm
