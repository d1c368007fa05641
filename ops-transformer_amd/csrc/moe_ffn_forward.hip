// The chain of the expert FFN behind one C entry (include/opapi_moe_ffn.h): host code only.
#include "opapi_moe_ffn.h"

#include <algorithm>

#include "aclnnop/aclnn_grouped_matmul_swiglu_quant.h"
#include "aclnnop/aclnn_grouped_matmul_v4.h"
#include "aclnnop/aclnn_moe_finalize_routing_v2.h"
#include "aclnnop/aclnn_moe_init_routing_v3.h"
#include "gemm_executor.h"
#include "moe_init_routing.h"
#include "opapi_common.h"

namespace {

constexpr int kTensors = 16;
enum { kX, kXScale, kExpertIdx, kTopKWeight, kW13, kW13Scale, kW2, kW2Scale, kExpandedX, kExpandedRowIdx, kCumsum, kExpandedScale, kH, kHScale, kY, kOut };

// The tensors of a packed array; false when it is too short or names more dimensions than a descriptor has.
bool Unpack(const int64_t* packed, uint64_t count, aclTensor (&tensors)[kTensors]) {
    uint64_t at = 1;
    for (aclTensor& t : tensors) {
        if (count < at + 3 || packed[at] < 0 || packed[at] > 8 || count < at + 3 + 2 * static_cast<uint64_t>(packed[at])) return false;
        const int64_t* const dims = packed + at + 3;
        const int64_t n = packed[at];
        t.dims.assign(dims, dims + n);
        t.strides.assign(dims + n, dims + 2 * n);
        t.storage = t.dims;
        t.dtype = static_cast<aclDataType>(packed[at + 1]);
        t.format = n == 5 ? ACL_FORMAT_FRACTAL_NZ : ACL_FORMAT_ND;
        t.data = reinterpret_cast<void*>(static_cast<uintptr_t>(packed[at + 2]));
        at += 3 + 2 * static_cast<uint64_t>(n);
    }
    return at == count;
}

struct Executors {
    aclOpExecutor* of[4] = {nullptr, nullptr, nullptr, nullptr};
    ~Executors() {  // those that no second phase has consumed
        for (aclOpExecutor* e : of) delete e;
    }
};

}  // namespace

extern "C" aclnnStatus opapiMoeFfnForward(const int64_t* packed, uint64_t count, void* workspace, uint64_t workspaceSize,
                                          aclrtStream stream, uint64_t* workspaceSizes, int32_t* enqueued,
                                          const char** failedOperator) try {
    using namespace opapi;
    ClearError();
    OPAPI_CHECK_NOTNULL(packed, "packed");
    OPAPI_CHECK_NOTNULL(workspaceSizes, "workspaceSizes");
    OPAPI_CHECK_NOTNULL(enqueued, "enqueued");
    OPAPI_CHECK_NOTNULL(failedOperator, "failedOperator");
    *enqueued = 0;
    *failedOperator = "opapiMoeFfnForward";
    std::fill(workspaceSizes, workspaceSizes + 5, 0);
    aclTensor t[kTensors];
    OPAPI_CHECK(count > 0 && (packed[0] == 2 || packed[0] == 3) && Unpack(packed, count, t), ACLNN_ERR_PARAM_INVALID,
                "opapiMoeFfnForward: the packed array holds no routing and sixteen tensors");
    const int64_t experts = t[kCumsum].dims.size() == 1 ? t[kCumsum].dims[0] : 0;
    // the lists do not own their tensors here: they are never passed to aclDestroyTensorList
    aclTensorList x, weight, scale, perToken, out;
    x.items = {&t[kH]};
    weight.items = {&t[kW2]};
    scale.items = {&t[kW2Scale]};
    perToken.items = {&t[kHScale]};
    out.items = {&t[kY]};

    Executors ex;
    aclnnStatus st;
    if (packed[0] == 3) {
        *failedOperator = "aclnnMoeInitRoutingV3GetWorkspaceSize";
        st = aclnnMoeInitRoutingV3GetWorkspaceSize(&t[kX], &t[kExpertIdx], &t[kXScale], nullptr, -1, 0, experts, 0, 0, true, -1, nullptr, 1,
                                                   &t[kExpandedX], &t[kExpandedRowIdx], &t[kCumsum], &t[kExpandedScale],
                                                   &workspaceSizes[0], &ex.of[0]);
    } else {
        *failedOperator = "aclnnMoeInitRoutingV2GetWorkspaceSize";
        st = PlanScaledRoutingV2(&t[kX], &t[kExpertIdx], &t[kXScale], experts, &t[kExpandedX], &t[kExpandedRowIdx], &t[kCumsum],
                                 &t[kExpandedScale], &workspaceSizes[0], &ex.of[0]);
    }
    if (st != ACLNN_SUCCESS) return st;
    *failedOperator = "aclnnGroupedMatmulSwigluQuantGetWorkspaceSize";
    st = aclnnGroupedMatmulSwigluQuantGetWorkspaceSize(&t[kExpandedX], &t[kW13], nullptr, nullptr, &t[kW13Scale], &t[kExpandedScale],
                                                       &t[kCumsum], &t[kH], &t[kHScale], nullptr, &workspaceSizes[1], &ex.of[1]);
    if (st != ACLNN_SUCCESS) return st;
    *failedOperator = "aclnnGroupedMatmulV4GetWorkspaceSize";
    st = aclnnGroupedMatmulV4GetWorkspaceSize(&x, &weight, nullptr, &scale, nullptr, nullptr, nullptr, &perToken, &t[kCumsum], nullptr,
                                              nullptr, nullptr, 3, 0, 0, 0, &out, nullptr, nullptr, &workspaceSizes[2], &ex.of[2]);
    if (st != ACLNN_SUCCESS) return st;
    *failedOperator = "aclnnMoeFinalizeRoutingV2GetWorkspaceSize";
    const bool weighted = !t[kTopKWeight].dims.empty() || t[kTopKWeight].data != nullptr;
    st = aclnnMoeFinalizeRoutingV2GetWorkspaceSize(&t[kY], &t[kExpandedRowIdx], nullptr, nullptr, nullptr,
                                                   weighted ? &t[kTopKWeight] : nullptr, nullptr, 2,
                                                   &t[kOut], &workspaceSizes[3], &ex.of[3]);
    if (st != ACLNN_SUCCESS) return st;
    const uint64_t largest = *std::max_element(workspaceSizes, workspaceSizes + 4);
    // One launch schedules both GEMMs where each has one: the down projection's table then waits behind everybody's workspace.  (A launch
    // of 4 us less: 1303 tokens top-2 of 8 experts, hidden and intermediate 1024, 67 -> 64 us; 1000 of these, 4096, 14336, 505 -> 500.)
    auto* const up = dynamic_cast<GemmExecutor*>(ex.of[1]);
    auto* const down = dynamic_cast<GemmExecutor*>(ex.of[2]);
    const uint64_t tableAt = AlignUp(largest, 256);
    const bool mayShare = up != nullptr && down != nullptr && up->stagingBytes == 0 && down->stagingBytes == 0 &&
                             gemm::SchedulesOnce(up->problem, up->plan) && gemm::SchedulesOnce(down->problem, down->plan);
    workspaceSizes[4] = mayShare ? tableAt + gemm::ScheduleBytes(down->plan) : largest;
    if (largest > workspaceSize) return ACLNN_SUCCESS;
    if (mayShare && workspaceSizes[4] <= workspaceSize) {  // (the second executor outlives the first one's run)
        down->shared.table = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + tableAt);
        up->shared.nextProblem = &down->problem;
        up->shared.nextPlan = &down->plan;
        up->shared.nextTable = down->shared.table;
    }

    static const char* const kRun[2][4] = {
        {"aclnnMoeInitRoutingV2", "aclnnGroupedMatmulSwigluQuant", "aclnnGroupedMatmulV4", "aclnnMoeFinalizeRoutingV2"},
        {"aclnnMoeInitRoutingV3", "aclnnGroupedMatmulSwigluQuant", "aclnnGroupedMatmulV4", "aclnnMoeFinalizeRoutingV2"}};
    for (int i = 0; i < 4; ++i) {
        *failedOperator = kRun[packed[0] == 3][i];
        aclOpExecutor* const executor = ex.of[i];
        ex.of[i] = nullptr;  // consumed, whatever the status
        st = RunAndRelease(workspace, workspaceSize, executor, stream);
        if (st != ACLNN_SUCCESS) return st;
    }
    *enqueued = 1;
    return ACLNN_SUCCESS;
} catch (...) {  // no exception may cross the C boundary
    opapi::SetError("out of host memory");
    return ACLNN_ERR_INNER;
}
