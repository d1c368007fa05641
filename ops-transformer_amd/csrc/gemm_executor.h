// What the executors of the two grouped-GEMM operators have in common, for the expert FFN's chain, which lets one launch schedule both.
#pragma once

#include "grouped_gemm_i8.h"
#include "opapi_common.h"

class GemmExecutor : public aclOpExecutor {
   public:
    gemm::Problem problem;
    gemm::Plan plan;
    gemm::SharedSchedule shared;
};
