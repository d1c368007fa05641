// Descriptor creation for callers that pay for every foreign call (the Python host): one flat array in, one call per
// tensor, and one call to release all tensors of an operator.  What they make and take are the handles of aclCreateTensor.
#pragma once

#include <stdint.h>

#include "acl/acl.h"

#ifdef __cplusplus
extern "C" {
#endif

// packed: number of dimensions n (at most 8), data type, address of the first element, n extents, n strides (in elements).
// The format is ND, the offset 0, the storage shape the view's.  Null where aclCreateTensor returns null.
ACL_API aclTensor* opapiCreateTensorPacked(const int64_t* packed);

ACL_API void opapiDestroyTensors(const aclTensor* const* tensors, uint64_t count);

// The first phase of an operator on descriptors that exist for the call only.  packed: the operator's number (0 aclnnMoeGatingTopKSoftmaxV2,
// 1 aclnnMoeInitRoutingV2, 2 aclnnMoeInitRoutingQuantV2, 3 aclnnMoeInitRoutingV3 on all experts, 4 aclnnGroupedMatmulSwigluQuant,
// 5 aclnnGroupedMatmulV4 on lists of one tensor, 6 aclnnMoeFinalizeRoutingV2), its scalars, then its tensors as above, both in the order of
// its first phase, absent tensors with no dimensions and no address.  Left out: offset and activeExpertRange of 3, outputOffset of 4, the
// lists of 5 other than x, weight, bias, scale, perTokenScale and out (the group list stands before out).
ACL_API aclnnStatus opapiPlanPacked(const int64_t* packed, uint64_t length, uint64_t* workspaceSize, aclOpExecutor** executor);

#ifdef __cplusplus
}
#endif
