// First phases on descriptors that travel in one packed array (include/opapi_descriptor.h): host code only.
#include "opapi_descriptor.h"

#include "aclnnop/aclnn_grouped_matmul_swiglu_quant.h"
#include "aclnnop/aclnn_grouped_matmul_v4.h"
#include "aclnnop/aclnn_moe_finalize_routing_v2.h"
#include "aclnnop/aclnn_moe_gating_top_k_softmax_v2.h"
#include "aclnnop/aclnn_moe_init_routing_quant_v2.h"
#include "aclnnop/aclnn_moe_init_routing_v2.h"
#include "aclnnop/aclnn_moe_init_routing_v3.h"
#include "opapi_common.h"

namespace {

// The operators by number, with how many scalars and tensors each takes.
enum { kGating, kRoutingV2, kRoutingQuantV2, kRoutingV3, kSwigluQuant, kGroupedMatmulV4, kFinalizeV2, kOperators };
constexpr int kScalars[kOperators] = {3, 6, 7, 8, 0, 4, 1};
constexpr int kTensors[kOperators] = {5, 6, 9, 7, 9, 7, 8};
constexpr int kMaxTensors = 9;

// Tensors from packed[at] on, count of them; absent ones (no dimensions, no address) stay null.  False when the array is not exactly theirs.
bool Unpack(const int64_t* packed, uint64_t at, uint64_t length, int count, aclTensor (&tensors)[kMaxTensors], aclTensor* (&given)[kMaxTensors]) {
    for (int i = 0; i < count; ++i) {
        if (length < at + 3 || packed[at] < 0 || packed[at] > 8 || length < at + 3 + 2 * static_cast<uint64_t>(packed[at])) return false;
        const int64_t n = packed[at];
        const int64_t* const dims = packed + at + 3;
        aclTensor& t = tensors[i];
        t.dims.assign(dims, dims + n);
        t.strides.assign(dims + n, dims + 2 * n);
        t.storage = t.dims;
        t.dtype = static_cast<aclDataType>(packed[at + 1]);
        t.data = reinterpret_cast<void*>(static_cast<uintptr_t>(packed[at + 2]));
        given[i] = n == 0 && t.data == nullptr ? nullptr : &t;
        at += 3 + 2 * static_cast<uint64_t>(n);
    }
    return at == length;
}

}  // namespace

extern "C" aclnnStatus opapiPlanPacked(const int64_t* packed, uint64_t length, uint64_t* workspaceSize, aclOpExecutor** executor) try {
    using namespace opapi;
    ClearError();
    OPAPI_CHECK_NOTNULL(packed, "packed");
    OPAPI_CHECK(length > 0 && packed[0] >= 0 && packed[0] < kOperators, ACLNN_ERR_PARAM_INVALID, "opapiPlanPacked: no such operator");
    const int op = static_cast<int>(packed[0]);
    aclTensor tensors[kMaxTensors];
    aclTensor* t[kMaxTensors] = {};
    OPAPI_CHECK(length >= 1 + static_cast<uint64_t>(kScalars[op]) &&
                    Unpack(packed, 1 + static_cast<uint64_t>(kScalars[op]), length, kTensors[op], tensors, t),
                ACLNN_ERR_PARAM_INVALID, "opapiPlanPacked: the packed array does not hold the operator's scalars and tensors");
    const int64_t* const s = packed + 1;
    switch (op) {
        case kGating:
            return aclnnMoeGatingTopKSoftmaxV2GetWorkspaceSize(t[0], t[1], s[0], s[1], s[2] != 0, t[2], t[3], t[4], workspaceSize, executor);
        case kRoutingV2:
            return aclnnMoeInitRoutingV2GetWorkspaceSize(t[0], t[1], s[0], s[1], s[2], s[3], s[4], s[5] != 0, t[2], t[3], t[4], t[5],
                                                         workspaceSize, executor);
        case kRoutingQuantV2:
            return aclnnMoeInitRoutingQuantV2GetWorkspaceSize(t[0], t[1], t[2], t[3], s[0], s[1], s[2], s[3], s[4], s[5] != 0, s[6], t[4], t[5],
                                                              t[6], t[7], t[8], workspaceSize, executor);
        case kRoutingV3:
            return aclnnMoeInitRoutingV3GetWorkspaceSize(t[0], t[1], t[2], nullptr, s[0], s[1], s[2], s[3], s[4], s[5] != 0, s[6], nullptr, s[7],
                                                         t[3], t[4], t[5], t[6], workspaceSize, executor);
        case kSwigluQuant:
            return aclnnGroupedMatmulSwigluQuantGetWorkspaceSize(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], nullptr, workspaceSize,
                                                                 executor);
        case kGroupedMatmulV4: {
            // one tensor a list, absent ones no list; the lists do not own their tensors here
            aclTensorList lists[7];
            aclTensorList* l[7] = {};
            for (int i = 0; i < 7; ++i) {
                if (t[i] == nullptr) continue;
                lists[i].items = {t[i]};
                l[i] = &lists[i];
            }
            return aclnnGroupedMatmulV4GetWorkspaceSize(l[0], l[1], l[2], l[3], nullptr, nullptr, nullptr, l[4], t[5], nullptr, nullptr, nullptr,
                                                        s[0], s[1], s[2], s[3], l[6], nullptr, nullptr, workspaceSize, executor);
        }
        default:
            return aclnnMoeFinalizeRoutingV2GetWorkspaceSize(t[0], t[1], t[2], t[3], t[4], t[5], t[6], s[0], t[7], workspaceSize, executor);
    }
} catch (...) {  // no exception may cross the C boundary
    opapi::SetError("out of host memory");
    return ACLNN_ERR_INNER;
}
