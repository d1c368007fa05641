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

#ifdef __cplusplus
}
#endif
