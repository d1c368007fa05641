"""Inner sizes off the 128-byte k-step on the LDS-ring kernels (K a multiple of 16, at least one k-step): the last k-step
overlaps the one before it and the overlap is multiplied by zero.  int32 and bf16 outputs bit-exact against the oracle,
SwiGLU-quant within one LSB."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["kmajor", "nd", "nz"])
@pytest.mark.parametrize("tile_m,K", [(32, 144), (64, 240), (64, 1040), (96, 160), (128, 208), (128, 1136), (160, 1120),
                                      (192, 144), (192, 1072), (256, 176), (256, 1088),
                                      (96, 1008), (192, 912), (256, 960)])
def test_k_off_the_step_grid(aclnn, oracle, dev, monkeypatch, tile_m, K, layout):
    """Overlaps of 16 to 112 bytes in every tile height and layout; K of eight
    steps (the fewest) and of nine is pulled where the height allows it.
    Several tiles per workgroup, an empty group, groups past a tile, and the tensors' last rows in the last tile."""
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", str(tile_m))
    rng = np.random.default_rng(tile_m + K)
    E, N = 40, 256 * 7 + 64
    sizes = rng.integers(0, 150, E)
    sizes[3] = 0
    sizes[-1] = 2 * tile_m + 5
    cumsum = np.cumsum(sizes).astype(np.int64)
    M = int(cumsum[-1])
    x = rng.integers(-127, 128, (M, K)).astype(np.int8)
    wt = rng.integers(-127, 128, (E, N, K)).astype(np.int8)
    scale = rng.uniform(1e-3, 1e-2, (E, N)).astype(np.float32)
    pt = rng.uniform(0.01, 0.1, M).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    w_dev = t(wt)
    if layout == "nz":
        w_nz = w_dev.view(E, N // 32, 32, K // 16, 16).permute(0, 1, 3, 4, 2).contiguous()
        wkw, wv, w = dict(weight_nz=(w_nz, "nz5d")), None, None
    else:
        w = w_dev.transpose(1, 2) if layout == "kmajor" else w_dev.transpose(1, 2).contiguous()
        wkw, wv = {}, [w]
    gl = t(cumsum)
    acc = aclnn.grouped_matmul_v4([t(x)], wv, group_list=gl, split_item=3, group_type=0, **wkw)[0]
    y = aclnn.grouped_matmul_v4([t(x)], wv, scale=[t(scale)], per_token_scale=[t(pt)], group_list=gl, split_item=3,
                                group_type=0, output_dtype=torch.bfloat16, **wkw)[0]
    q, qs = aclnn.grouped_matmul_swiglu_quant(t(x), w, gl, t(scale), t(pt), **wkw)
    torch.cuda.synchronize()
    assert np.array_equal(acc.cpu().numpy(), oracle.grouped_matmul_i32(x, wt, cumsum, w_trans=True))
    ref = oracle.grouped_matmul_dequant(x, wt, scale, pt, cumsum, w_trans=True, out_dtype=oracle.DT_BF16)
    assert np.array_equal(y.view(torch.int16).cpu().numpy().view(np.uint16), ref)
    q_ref, qs_ref = oracle.grouped_matmul_swiglu_quant(x, wt, scale, pt, cumsum, w_trans=True)
    diff = np.abs(q.cpu().numpy().astype(np.int32) - q_ref.astype(np.int32))
    assert diff.max() <= 1 and (diff != 0).mean() < 1e-3
    np.testing.assert_allclose(qs.cpu().numpy(), qs_ref, rtol=1e-5)
