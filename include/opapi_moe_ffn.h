// One pass of the quantized expert FFN as one call: the first phases of
//   aclnnMoeInitRoutingV2 (or V3) -> aclnnGroupedMatmulSwigluQuant -> aclnnGroupedMatmulV4 -> aclnnMoeFinalizeRoutingV2
// on descriptors made from one packed array, then their second phases on one workspace.  No counterpart in the reference,
// whose callers chain the operators themselves.  For hosts that pay for every foreign call: a pass over a few rows takes the
// device 45 us, and thirty descriptors and ten calls from Python took longer than that (one token over 128 experts, hidden 4096,
// intermediate 1536: 64.6 -> 46.0 us a pass; 256 tokens over 8 experts of 1024 x 1024: 64.4 -> 33.2).
// Validation, plans, kernels and results are those of the operators, with one difference in how the rows are routed behind V2:
// the per-token scales are copied along with the rows instead of being routed by a second call of the operator.
#pragma once

#include <stdint.h>

#include "acl/acl.h"

#ifdef __cplusplus
extern "C" {
#endif

// packed: routing (2 or 3), then sixteen tensors, each as opapiCreateTensorPacked takes it (number of dimensions, data type,
// address, extents, strides), in the order
//   x int8 [T, H], xScale fp32 [T], expertIdx int32 [T, K], weights of the combine [T, K] (no dimensions at address 0: none, K 1),
//   w13 [E, H, 2I], w13Scale [E, 2I], w2 [E, I, H], w2Scale [E, H]  (a five-dimensional weight is FRACTAL_NZ),
//   expandedX, expandedRowIdx, cumsum, expandedScale, h, hScale, y, out.
// count: values in the array.  workspaceSizes[5]: what each operator asks for, and what the pass makes use of, which is the largest of
// these and, where one launch can schedule both GEMMs, room behind it for the second one's table.  When the largest is more
// than workspaceSize nothing is enqueued and ACLNN_SUCCESS is returned with *enqueued 0: call again with workspaceSizes[4] bytes.  With
// the largest but less than those every GEMM is scheduled by a launch of its own, with the same results.
// On failure *failedOperator names the entry point that returned the status (its message: aclGetRecentErrMsg).
ACL_API aclnnStatus opapiMoeFfnForward(const int64_t* packed, uint64_t count, void* workspace, uint64_t workspaceSize, aclrtStream stream,
                                       uint64_t* workspaceSizes, int32_t* enqueued, const char** failedOperator);

#ifdef __cplusplus
}
#endif
