// Expert-grouped int8 GEMM for a handful of rows per expert: the SwiGLU kernels (see grouped_gemm_i8_slim.h).
#include "grouped_gemm_i8_slim.h"

namespace gemm {

hipError_t LaunchSlimSwiglu(const Plan& plan, const KernelArgs& args, const SlimList& list, hipStream_t stream) {
    return LaunchSlimLayout<true>(plan, args, list, stream);
}

}  // namespace gemm
