// First phase of aclnnMoeInitRoutingV2 (dropless, int32 cumsum) that also copies a per-token scale [T] fp32 along with the rows,
// as aclnnMoeInitRoutingV3 does (defined in moe_init_routing.hip).
#pragma once

#include <cstdint>

#include "acl/acl.h"

namespace opapi {

aclnnStatus PlanScaledRoutingV2(const aclTensor* x, const aclTensor* expertIdx, const aclTensor* xScale, int64_t expertNum,
                                const aclTensor* expandedX, const aclTensor* expandedRowIdx, const aclTensor* cumsum,
                                const aclTensor* expandedScale, uint64_t* workspaceSize, aclOpExecutor** executor);

}  // namespace opapi
