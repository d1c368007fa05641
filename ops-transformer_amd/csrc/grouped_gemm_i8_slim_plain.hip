// Expert-grouped int8 GEMM for a handful of rows per expert: the int32 and dequantising kernels (see grouped_gemm_i8_slim.h).
#include "grouped_gemm_i8_slim.h"

namespace gemm {

hipError_t LaunchSlimPlain(const Plan& plan, const KernelArgs& args, const SlimList& list, hipStream_t stream) {
    return LaunchSlimLayout<false>(plan, args, list, stream);
}

}  // namespace gemm
