"""The one-call expert FFN (opapiMoeFfnForward, what MoeFfnW8A8.forward runs): what it refuses, on the CPU, and on the GPU that
its results are those of the four operators called one by one."""
import ctypes
import os
import struct
import subprocess
import sys

import pytest
import torch


def _call(aclnn, data, workspace=None, nbytes=0):
    sizes = (ctypes.c_uint64 * 5)()
    enqueued, failed = ctypes.c_int32(-1), ctypes.c_char_p(None)
    st = aclnn.lib().opapiMoeFfnForward(data, len(data) // 8, workspace, nbytes, None, sizes, ctypes.byref(enqueued), ctypes.byref(failed))
    return st, list(sizes), enqueued.value, (failed.value or b"").decode()


def _tensors(T, H, I, E, K, v3=False, dev="cpu"):
    M = T * K
    i8 = lambda *s: torch.zeros(s, dtype=torch.int8, device=dev)
    f = lambda *s: torch.zeros(s, device=dev)
    return [i8(T, H), f(T), torch.zeros((T, K), dtype=torch.int32, device=dev), f(T, K), i8(E, 2 * I, H).transpose(1, 2), f(E, 2 * I),
            i8(E, H, I).transpose(1, 2), f(E, H), i8(M, H), torch.zeros(M, dtype=torch.int32, device=dev),
            torch.zeros(E, dtype=torch.int64 if v3 else torch.int32, device=dev), f(M), i8(M, I), f(M),
            torch.zeros((M, H), dtype=torch.bfloat16, device=dev), torch.zeros((T, H), dtype=torch.bfloat16, device=dev)]


def _pack(aclnn, routing, tensors):
    return struct.pack("q", routing) + b"".join(aclnn._packed(t) for t in tensors)


@pytest.mark.parametrize("routing", [2, 3])
def test_too_small_a_workspace_enqueues_nothing(aclnn, routing):
    st, sizes, enqueued, _ = _call(aclnn, _pack(aclnn, routing, _tensors(4, 128, 64, 4, 2, routing == 3)))
    assert st == 0 and enqueued == 0
    assert sizes[0] > 0 and sizes[1] > 0 and sizes[4] == max(sizes[:4])


@pytest.mark.parametrize("cap_mb,shared", [(None, True), (1, False)])  # 1 MB: the SwiGLU operator runs in bands, each with its schedule
def test_one_schedule_adds_the_second_table(aclnn, monkeypatch, cap_mb, shared):
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    monkeypatch.delenv("OPAPI_SWIGLU_WORKSPACE_MB", raising=False)
    if cap_mb:
        monkeypatch.setenv("OPAPI_SWIGLU_WORKSPACE_MB", str(cap_mb))
    st, sizes, enqueued, _ = _call(aclnn, _pack(aclnn, 2, _tensors(2000, 1024, 512, 4, 2, False)))
    assert st == 0 and enqueued == 0
    assert (sizes[4] > max(sizes[:4])) == shared and sizes[4] - max(sizes[:4]) <= sizes[2] + 256


@pytest.mark.parametrize("routing", [2, 3])
def test_a_pass_that_was_not_enqueued_is_an_error(aclnn, monkeypatch, routing):
    """The outputs are reused from pass to pass: returning without having enqueued one would hand out the last one's."""
    class NeverGrows(aclnn.Workspace):
        def reserve(self, nbytes, device, api=None):
            return None
    monkeypatch.setattr(aclnn, "_stream_ptr", lambda: None)
    with pytest.raises(aclnn.AclnnError, match="workspace"):
        aclnn.moe_ffn_forward(routing, _tensors(4, 128, 64, 4, 2, routing == 3), NeverGrows(), "cpu")


def test_malformed_arrays_are_refused(aclnn):
    good = _pack(aclnn, 2, _tensors(4, 128, 64, 4, 2))
    bad_rank = bytearray(good)
    bad_rank[8:16] = struct.pack("q", 9)
    negative_rank = bytearray(good)
    negative_rank[8:16] = struct.pack("q", -1)
    for data in (b"", struct.pack("q", 2), good[:-8], good + b"\0" * 8, struct.pack("q", 1) + good[8:], bytes(bad_rank), bytes(negative_rank)):
        st, _, enqueued, name = _call(aclnn, data)
        assert st == aclnn.ACLNN_ERR_PARAM_INVALID and enqueued == 0 and name == "opapiMoeFfnForward"
    assert _call(aclnn, good)[0] == 0


@pytest.mark.parametrize("which,replacement,operator", [
    (0, torch.zeros((5, 128), dtype=torch.int8), "aclnnMoeInitRoutingV2GetWorkspaceSize"),
    (1, torch.zeros(4, dtype=torch.float16), "aclnnMoeInitRoutingV2GetWorkspaceSize"),
    (1, torch.zeros(5), "aclnnMoeInitRoutingV2GetWorkspaceSize"),
    (11, torch.zeros(7), "aclnnMoeInitRoutingV2GetWorkspaceSize"),
    (5, torch.zeros((4, 64)), "aclnnGroupedMatmulSwigluQuantGetWorkspaceSize"),
    (14, torch.zeros((8, 64), dtype=torch.bfloat16), "aclnnGroupedMatmulV4GetWorkspaceSize"),
    (15, torch.zeros((4, 64), dtype=torch.bfloat16), "aclnnMoeFinalizeRoutingV2GetWorkspaceSize")])
def test_each_operator_still_checks_its_tensors(aclnn, which, replacement, operator):
    tensors = _tensors(4, 128, 64, 4, 2)
    tensors[which] = replacement
    st, _, enqueued, name = _call(aclnn, _pack(aclnn, 2, tensors))
    assert st != 0 and enqueued == 0 and name == operator and aclnn.last_error()


FAILING_NEW = """
#include <cstdlib>
#include <new>
static thread_local long left = -1;  // allocations until the one that fails; negative: none does
extern "C" void fail_new_after(long n) { left = n; }
void* operator new(std::size_t n) {
    if (left >= 0 && left-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
"""

CHILD = """
import ctypes, sys
sys.path[:0] = [{root!r}, {tests!r}]
from __graft_entry__ import load_package
import test_moe_ffn_forward as t
aclnn = load_package().aclnn
arm = ctypes.CDLL({lib!r}).fail_new_after
arm.argtypes = [ctypes.c_long]
for routing in (2, 3):
    data = t._pack(aclnn, routing, t._tensors(4, 128, 64, 4, 2, routing == 3))
    aclnn.lib()
    for n in range(10000):
        arm(n)
        st, _, enqueued, _ = t._call(aclnn, data)
        arm(-1)
        assert enqueued == 0
        if st == 0:
            break
    print("survived", routing, n)
    assert n > 16
"""


def test_running_out_of_host_memory_is_a_status(tmp_path):
    """Every allocation of the call in turn fails: no exception leaves the C entry (it would end the process)."""
    src, lib = tmp_path / "failing_new.cpp", tmp_path / "libfailing_new.so"
    src.write_text(FAILING_NEW)
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", str(src), "-o", str(lib)])
    tests = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, LD_PRELOAD=":".join([str(lib)] + [p for p in [os.environ.get("LD_PRELOAD")] if p]))
    res = subprocess.run([sys.executable, "-c", CHILD.format(root=os.path.dirname(tests), tests=tests, lib=str(lib))], env=env,
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert res.returncode == 0 and res.stdout.count("survived") == 2, res.stdout[-2000:]


def test_weights_of_the_combine_may_be_absent(aclnn):
    """As with the operator itself: one expert per token, unweighted.  Without them a row of more experts has nowhere to go."""
    for K, ok in ((1, True), (2, False)):
        tensors = _tensors(4, 128, 64, 4, K)
        tensors[3] = None
        st, sizes, enqueued, name = _call(aclnn, _pack(aclnn, 2, tensors))
        assert (st == 0) == ok and enqueued == 0 and name == "aclnnMoeFinalizeRoutingV2GetWorkspaceSize"


@pytest.mark.gpu
def test_top_1_without_weights(pkg, dev):
    g = torch.Generator(device=dev).manual_seed(1)
    i8 = lambda *s: torch.empty(s, dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    f = lambda *s: torch.rand(s, device=dev, generator=g) * 0.01 + 1e-3
    ffn = pkg.MoeFfnW8A8(i8(4, 256, 256), f(4, 256), i8(4, 256, 128), f(4, 256))
    xq, xs, idx = i8(9, 256), f(9), torch.randint(0, 4, (9, 1), device=dev, generator=g, dtype=torch.int32)
    want = ffn.forward(xq, xs, idx, torch.ones((9, 1), device=dev)).clone()
    assert torch.equal(ffn.forward(xq, xs, idx, None), want) and want.any()


@pytest.mark.gpu
@pytest.mark.parametrize("routing", ["v2", "v3"])
@pytest.mark.parametrize("tokens", [1, 3, 257, 1300])
def test_equals_the_operators_one_by_one(pkg, aclnn, dev, tokens, routing):
    H, I, E, K = 256, 128, 8, 3
    g = torch.Generator(device=dev).manual_seed(tokens)
    i8 = lambda *s: torch.empty(s, dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    f = lambda *s: torch.rand(s, device=dev, generator=g) * 0.01 + 1e-3
    w13, w2, w13s, w2s, xq = i8(E, 2 * I, H), i8(E, H, I), f(E, 2 * I), f(E, H), i8(tokens, H)
    xs = f(tokens, 2)[:, 1] if routing == "v2" else f(tokens)  # a strided column of scales
    idx = torch.rand((tokens, E), device=dev, generator=g).topk(K, dim=1)[1].int()
    wgt = f(tokens, K)
    got = pkg.MoeFfnW8A8(w13, w13s, w2, w2s, routing=routing).forward(xq, xs, idx, wgt)
    ex, row_idx, cumsum, _ = aclnn.moe_init_routing_v2(xq, idx, 0, 0, E, 0, 1, False)
    es, _, _, _ = aclnn.moe_init_routing_v2(xs.contiguous().view(tokens, 1), idx, 0, 0, E, 0, 0, False)
    h, hs = aclnn.grouped_matmul_swiglu_quant(ex, w13.transpose(1, 2), cumsum, w13s, es.view(-1))
    y = aclnn.grouped_matmul_v4([h], [w2.transpose(1, 2)], scale=[w2s], per_token_scale=[hs], group_list=cumsum, split_item=3,
                                group_type=0, group_list_type=0, output_dtype=torch.bfloat16)[0]
    want = aclnn.moe_finalize_routing_v2(y, row_idx, scales=wgt, drop_pad_mode=2)
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_a_workspace_without_room_for_the_second_table(aclnn, dev):
    """The largest of the operators' sizes is enough: the pass is enqueued, with the results of one that has room for both tables."""
    T, H, I, E, K = 2000, 1024, 512, 4, 2
    tensors = _tensors(T, H, I, E, K, dev=dev)
    g = torch.Generator(device=dev).manual_seed(2)
    for t in tensors[:8]:
        if t.dtype == torch.int8:
            t.random_(-127, 128, generator=g)
        elif t.dtype == torch.float32:
            t.uniform_(1e-3, 1e-2, generator=g)
    tensors[2].copy_(torch.rand((T, E), device=dev, generator=g).topk(K, dim=1)[1])
    data = _pack(aclnn, 2, tensors)
    sizes = _call(aclnn, data)[1]
    assert sizes[4] > max(sizes[:4])
    outs = []
    for nbytes in (sizes[4], sizes[4] - 1, max(sizes[:4])):
        workspace = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        tensors[15].zero_()
        torch.cuda.synchronize()
        st, _, enqueued, name = _call(aclnn, data, workspace.data_ptr(), nbytes)
        torch.cuda.synchronize()
        assert st == 0 and enqueued == 1, name
        outs.append(tensors[15].clone())
    assert outs[0].any() and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert _call(aclnn, data, 0x1000, max(sizes[:4]) - 1)[1:3] == (sizes, 0)
