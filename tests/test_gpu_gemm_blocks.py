"""The ring GEMM kernels where their tiles end: row counts around the 16-row blocks and the 256-row tile, channel counts around
a lane's vector of four and a tile's 256, launches of at most one tile per workgroup and of one more, in the three weight
layouts and with every output type, against exact integer products (float64) and the epilogue's own fp32 arithmetic."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(w_enk, layout):
    """(weight view, weight_nz) of K-contiguous int8 storage [E, N, K]."""
    if layout == "nz":
        E, N, K = w_enk.shape
        return None, (w_enk.view(E, N // 32, 32, K // 16, 16).permute(0, 1, 3, 4, 2).contiguous(), "nz5d")
    view = w_enk.transpose(1, 2)
    return (view.contiguous() if layout == "nd" else view), None


def _run(aclnn, sizes, N, K, layout, out_dtype, seed, offset=0, kind="cumsum"):
    """offset: values in front of the output in its buffer (and sixteen behind it), which no store may touch."""
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(seed)
    E, M = len(sizes), sum(sizes)
    x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    w = torch.randint(-127, 128, (E, N, K), generator=g, dtype=torch.int8)
    scale = torch.rand((E, N), generator=g) * 0.01 + 1e-3
    row_scale = torch.rand((M,), generator=g) * 0.05 + 1e-2
    if kind == "sparse":  # pairs in falling order of the experts, those without rows left out
        order = [e for e in reversed(range(E)) if sizes[e] > 0]
        listed = torch.tensor([[e, sizes[e]] for e in order] + [[0, 0]] * (E - len(order)))
    else:
        order = list(range(E))
        listed = torch.cumsum(torch.tensor(sizes), 0) if kind == "cumsum" else torch.tensor(sizes)
    listed = listed.int() if kind == "counts32" else listed
    acc = torch.empty((M, N), dtype=torch.float64)
    begin = 0
    for e in order:
        n = sizes[e]
        acc[begin:begin + n] = x[begin:begin + n].double() @ w[e].double().t()
        begin += n
    buffer = torch.full((offset + M * N + 16,), 7, dtype=out_dtype, device=dev)
    out = buffer[offset:offset + M * N].view(M, N)
    view, nz = _weights(w.to(dev), layout)
    scales = {} if out_dtype == torch.int32 else {"scale": [scale.to(dev)], "per_token_scale": [row_scale.to(dev)]}
    aclnn.grouped_matmul_v4([x.to(dev)], None if view is None else [view], weight_nz=nz, group_list=listed.to(dev), split_item=3,
                            group_type=0, group_list_type={"cumsum": 0, "sparse": 2}.get(kind, 1), out=[out], **scales)
    assert (buffer[:offset] == 7).all() and (buffer[offset + M * N:] == 7).all()
    if out_dtype == torch.int32:
        return out.cpu(), acc.to(torch.int32)
    group = torch.repeat_interleave(torch.tensor(order), torch.tensor([sizes[e] for e in order]))
    return out.cpu(), ((acc.float() * scale[group]) * row_scale[:, None]).to(out_dtype)


# rows of the groups: around a 16-row block, the 32 rows of a wave-row pair, and the tallest tile
ROWS = {"blocks": [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65], "tile": [255, 0, 256, 257, 271, 272, 273]}


@pytest.mark.parametrize("out_dtype", [torch.int32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", sorted(ROWS))
@pytest.mark.parametrize("height", [32, 96, 160, 192, 256])
def test_row_remainders(aclnn, monkeypatch, height, rows, out_dtype):
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", str(height))
    got, want = _run(aclnn, ROWS[rows], 512, 256, "k", out_dtype, height)
    assert torch.equal(got, want)


@pytest.mark.parametrize("out_dtype", [torch.int32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout,N", [("k", 4), ("k", 30), ("k", 62), ("k", 66), ("k", 257), ("k", 258), ("k", 260), ("nd", 16),
                                      ("nd", 144), ("nd", 272), ("nz", 32), ("nz", 96), ("nz", 288)])
def test_channel_remainders(aclnn, monkeypatch, layout, N, out_dtype):
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "128")
    got, want = _run(aclnn, [100, 0, 37, 130], N, 384, layout, out_dtype, N)
    assert torch.equal(got, want)


@pytest.mark.parametrize("out_dtype", [torch.int32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [[20, 0, 17], [100, 0, 37, 130]])  # the byte-wise kernel's tiles of 32 and of 128 rows
@pytest.mark.parametrize("layout,N,K", [("k", 30, 100), ("k", 257, 1001), ("k", 258, 100), ("nd", 33, 100), ("nd", 258, 333), ("nz", 288, 64)])
def test_bytewise_channel_remainders(aclnn, monkeypatch, layout, N, K, sizes, out_dtype):
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    got, want = _run(aclnn, sizes, N, K, layout, out_dtype, N)
    assert torch.equal(got, want)


@pytest.mark.parametrize("layout", ["k", "nd", "nz"])
@pytest.mark.parametrize("out_dtype,offset", [(torch.bfloat16, 1), (torch.bfloat16, 2), (torch.float16, 4), (torch.int32, 1), (torch.int32, 2)])
@pytest.mark.parametrize("N", [512, 514, 516])
def test_outputs_off_the_vector_grid(aclnn, monkeypatch, N, out_dtype, offset, layout):
    """Vectors of two and four dwords that begin on a dword: views into a buffer, and rows of 4k + 2 channels."""
    N = {"k": N, "nd": 512, "nz": 512}[layout]
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "128")
    got, want = _run(aclnn, [100, 0, 37, 130], N, 256, layout, out_dtype, N, offset)
    assert torch.equal(got, want)


@pytest.mark.parametrize("out_dtype", [torch.int32, torch.bfloat16])
@pytest.mark.parametrize("layout,N", [("nd", 272), ("nz", 288)])
@pytest.mark.parametrize("height,K", [(32, 128), (32, 400), (64, 256), (64, 1040), (256, 144)])
def test_channels_side_by_side_at_every_depth(aclnn, monkeypatch, height, K, layout, N, out_dtype):
    """Weights whose channels are neighbours in memory: fewer k-steps than the ring has stages, more, and a masked last one."""
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", str(height))
    got, want = _run(aclnn, [20, 0, 17, 64, 33], N, K, layout, out_dtype, K)
    assert torch.equal(got, want)


@pytest.mark.parametrize("height,groups,N,K", [(32, 400, 1024, 128), (64, 200, 4096, 384)])
def test_shares_of_more_tiles_than_the_ring_holds(aclnn, monkeypatch, height, groups, N, K):
    """1600 and 3200 small tiles: seven and thirteen to a workgroup, of which six are decoded ahead."""
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", str(height))
    got, want = _run(aclnn, [1, 3] * (groups // 2), N, K, "k", torch.bfloat16, K)
    assert torch.equal(got, want)


# Groups alike, one m-tile each, eight n-tiles: whole rounds of tiles dealt out, with nothing behind them, one group's tiles, and a part of
# a round that is drawn; one group in twelve of other rows, more than a tile's, and all rounds but two are drawn
@pytest.mark.parametrize("height", [96, 192])
@pytest.mark.parametrize("groups,odd", [(96, 70), (97, 70), (131, 70), (131, 260)])
def test_even_groups_and_uneven_ones(aclnn, monkeypatch, groups, odd, height):
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", str(height))
    got, want = _run(aclnn, [odd if e % 12 == 5 else 70 for e in range(groups)], 2048, 1024, "k", torch.bfloat16, groups)
    assert torch.equal(got, want)


@pytest.mark.parametrize("groups,height", [(128, 256), (129, 256), (192, 192)])
def test_one_round_of_pulled_tiles_and_one_more(aclnn, monkeypatch, groups, height):
    """Two n-tiles per group: 256 and 258 tiles of 256 rows (256 workgroups), and 384 of 192."""
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", str(height))
    got, want = _run(aclnn, [80] * groups, 512, 1024, "k", torch.int32, groups)
    assert torch.equal(got, want)


# Launches of few tiles, which the scheduling kernel may cut lower than planned, and each group evenly: groups around one and two low
# tiles, around a short even tile and one of ten (ten even tiles of 1441 rows are nine rows short of the tenth), idle groups, and
# (four of 250 rows beside 64 n-tiles: two rounds instead of one) a launch that stays as it is.  With half the channels ("narrow") only
# row-major weights take this path: the other layouts' 64-row tiles of the kernels for a handful of rows are one round.
FEW = {"even": ([250] * 8, 1024), "uneven": ([161, 0, 320, 321, 64, 65, 160, 1], 2048), "many": ([1441, 1760, 7], 1024), "tall": ([250] * 4, 16384),
       "uneven_narrow": ([161, 0, 320, 321, 64, 65, 160, 1], 1024), "many_narrow": ([1441, 1760, 7], 512)}


def _few_rows(name, layout):
    return 256 if name == "tall" else 64 if name.endswith("narrow") and layout != "nd" else 160


def _spanned(aclnn, call):
    """(what call returns, rows of the ring kernels' tallest tiles in it)"""
    aclnn.gemm_workgroup_spans_enable(True)
    try:
        result = call()
        spans = aclnn.gemm_workgroup_spans_report()
    finally:
        aclnn.gemm_workgroup_spans_enable(False)
    assert len(spans) == 1
    return result, next(iter(spans.values()))["tile_rows"]


@pytest.mark.parametrize("layout,K", [("k", 1024), ("k", 1040), ("nd", 1024), ("nz", 1040)])
@pytest.mark.parametrize("name", sorted(FEW))
def test_few_tiles(aclnn, monkeypatch, name, layout, K):
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    sizes, N = FEW[name]
    (got, want), rows = _spanned(aclnn, lambda: _run(aclnn, sizes, N, K, layout, torch.bfloat16, K))
    assert rows == _few_rows(name, layout)
    assert torch.equal(got, want)


@pytest.mark.parametrize("layout", ["k", "nd"])
@pytest.mark.parametrize("kind", ["counts", "counts32", "sparse"])
def test_few_tiles_of_other_lists(aclnn, monkeypatch, kind, layout):
    """The even cut on counts and on (expert, rows) pairs, whose groups lie in the order of the list."""
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    sizes, N = FEW["uneven"]
    (got, want), rows = _spanned(aclnn, lambda: _run(aclnn, sizes, N, 1024, layout, torch.bfloat16, 3, kind=kind))
    assert rows == 160
    assert torch.equal(got, want)


@pytest.mark.parametrize("bands", [False, True])
@pytest.mark.parametrize("layout", ["k", "nd"])
@pytest.mark.parametrize("name", sorted(FEW))
def test_few_tiles_swiglu_equals_a_forced_height(aclnn, oracle, dev, monkeypatch, name, layout, bands):
    """Every row against the same call at a forced height (S and its row maximum do not depend on how the rows are cut into tiles), rows
    at the ends of groups and tiles against the oracle.  bands: S for one band of rows at a time, each cut by itself."""
    sizes, N = FEW[name]
    K, E, M = 1024, len(sizes), sum(sizes)
    monkeypatch.delenv("OPAPI_SWIGLU_WORKSPACE_MB", raising=False)
    if bands:
        monkeypatch.setenv("OPAPI_SWIGLU_WORKSPACE_MB", str(max(1, 512 * N * 2 >> 20)))  # 512 rows
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.empty((M, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    w_enk = torch.empty((E, N, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    w = w_enk.transpose(1, 2).contiguous() if layout == "nd" else w_enk.transpose(1, 2)
    scale, x_scale = torch.rand((E, N), device=dev, generator=g) * 1e-3, torch.rand((M,), device=dev, generator=g) * 1e-2
    cumsum = torch.cumsum(torch.tensor(sizes), 0).to(dev)
    call = lambda: aclnn.grouped_matmul_swiglu_quant(x, w, cumsum, scale, x_scale)
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    (y, ys), rows = _spanned(aclnn, call)  # of the last band
    # (a launch that runs in bands is none of a handful of rows, and the second band of the tall one is small)
    assert rows == (160 if bands else _few_rows(name, layout))
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "256")
    (y256, ys256), rows = _spanned(aclnn, call)
    assert rows == 256 and torch.equal(y, y256) and torch.equal(ys, ys256)
    begins = [sum(sizes[:e]) for e in range(E)]
    sample = sorted({b + r for b, n in zip(begins, sizes) for r in (0, 15, 16, 79, 80, 127, 128, 159, 160, 255, 256, n - 1) if r < n})[:60]
    h, hs = oracle.grouped_matmul_swiglu_quant(x.cpu().numpy(), w_enk.cpu().numpy(), scale.cpu().numpy(), x_scale.cpu().numpy(),
                                               cumsum.cpu().numpy(), w_trans=True, rows=np.array(sample))
    diff = np.abs(y.cpu().numpy()[sample].astype(np.int32) - h.astype(np.int32))
    assert diff.max() <= 1 and (diff != 0).mean() < 1e-3  # an LSB where exp and division round differently
    np.testing.assert_allclose(ys.cpu().numpy()[sample], hs, rtol=1e-5)


# Groups whose sizes the scheduling kernel looks at: alike (one geometry: for SwiGLU tiles of two times 256 channels), one that needs a
# second m-tile (no wide tiles), and nearly all of at most 64 rows (two geometries).  N: whole pairs of 256 channels, a second 256
# that begin over the first's, a last tile of 256.
SIZES = {"alike": ([65, 80, 96, 97, 128, 129, 159, 160, 1, 0, 64, 100, 112, 144, 145, 81] * 8, 160),
         "over": ([65, 80, 96, 97, 70, 81, 112, 160] * 15 + [0, 100, 100, 100, 100, 100, 161, 100], 192),
         "small": ([60, 64, 63, 49, 48, 33, 64, 64] * 15 + [60, 64, 64, 64, 160, 160, 159, 250], 192)}


@pytest.mark.parametrize("layout,K,columns", [("k", 1280, 1024), ("k", 1296, 1001), ("k", 1536, 880), ("nd", 1280, 1008), ("nz", 1296, 992)])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_tiles_by_sizes_swiglu_equals_a_forced_height(aclnn, dev, monkeypatch, name, layout, K, columns):
    sizes, want_rows = SIZES[name]
    E, M = len(sizes), sum(sizes)
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.empty((M, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    w = torch.empty((E, 2 * columns, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    view, nz = _weights(w, layout)
    scale, x_scale = torch.rand((E, 2 * columns), device=dev, generator=g) * 1e-3, torch.rand((M,), device=dev, generator=g) * 1e-2
    cumsum = torch.cumsum(torch.tensor(sizes), 0).to(dev)

    def call():
        out = (torch.full((M, columns), 7, dtype=torch.int8, device=dev), torch.full((M,), 7.0, device=dev))
        return aclnn.grouped_matmul_swiglu_quant(x, view, cumsum, scale, x_scale, out=out, weight_nz=nz)

    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    (y, ys), rows = _spanned(aclnn, call)
    assert rows == want_rows
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "96")
    (y96, ys96), rows = _spanned(aclnn, call)
    assert rows == 96 and torch.equal(y, y96) and torch.equal(ys, ys96)


@pytest.mark.parametrize("layout,K", [("k", 1024), ("nd", 1040), ("nz", 1152)])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_tiles_by_sizes_down(aclnn, monkeypatch, name, layout, K):
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    sizes, want_rows = SIZES[name]
    (got, want), rows = _spanned(aclnn, lambda: _run(aclnn, sizes, 2208, K, layout, torch.bfloat16, K))
    assert rows == (160 if name == "over" else want_rows)  # (one group in 128 with a small second m-tile)
    assert torch.equal(got, want)


# 130 rows per group: even ones take wide tiles of 160 rows, uneven ones 192, of which these lists need more than M / 256 beyond one per group
@pytest.mark.parametrize("sizes", [[193] * 86 + [1] * 42, [2080] * 7 + [17] * 98 + [18] * 23])
def test_table_holds_lists_of_many_second_tiles(aclnn, dev, monkeypatch, sizes):
    K, columns, E, M = 1280, 1024, len(sizes), sum(sizes)
    assert (E, M) == (128, 130 * 128) and sum((r + 191) // 192 for r in sizes) > M // 256 + E
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.empty((M, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    w = torch.empty((E, 2 * columns, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    scale, x_scale = torch.rand((E, 2 * columns), device=dev, generator=g) * 1e-3, torch.rand((M,), device=dev, generator=g) * 1e-2
    cumsum = torch.cumsum(torch.tensor(sizes), 0).to(dev)

    def call():
        out = (torch.full((M, columns), 7, dtype=torch.int8, device=dev), torch.full((M,), 7.0, device=dev))
        return aclnn.grouped_matmul_swiglu_quant(x, w.transpose(1, 2), cumsum, scale, x_scale, out=out)

    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    (y, ys), rows = _spanned(aclnn, call)
    assert rows == 192
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "96")
    (y96, ys96), rows = _spanned(aclnn, call)
    assert rows == 96 and torch.equal(y, y96) and torch.equal(ys, ys96)


# What else the sizes decide: 64-row tiles for all, dealt out with a part of a round; the big tiles of two geometries, 96 and 192 of them all begun
# with and 304 that are not; wide tiles beside second m-tiles, in more than four rounds and in most of one; rows of weights that begin inside
# cache lines, K-contiguous and row-major, in launches of few and of many k-steps a workgroup
FORMS = {"dealt": ([30, 29, 33, 64, 1, 28, 35, 31] * 15 + [65, 70, 129, 0, 30, 30, 17, 30], "k", 1280, 1024, 64),
         "dealt_blocked": ([30, 29, 33, 64, 1, 28, 35, 31] * 15 + [65, 70, 129, 0, 30, 30, 17, 30], "nz", 1280, 1024, 64),
         "begun": ([25] * 120 + [64, 0, 1, 1] + [1150] * 4, "k", 1280, 1024, 192),
         "begun_long": ([14] * 120 + [64, 0, 1, 1] + [575] * 4, "k", 4096, 1024, 192),
         "some_begun": ([13] * 120 + [192 * 4, 300, 700, 192 * 5, 192 * 5, 192 * 5, 1100, 1300], "k", 1280, 1024, 192),
         "wide_over": ([100] * 230 + [161, 200, 320, 321, 65] * 5, "k", 1024, 1024, 160),
         "wide_round": ([80] * 26 + [200, 161, 170, 180, 190, 320], "k", 4096, 1536, 160),
         "short": ([50] * 100 + [161, 200] * 6 + [70] * 16, "k", 1296, 1024, 160),
         "long": ([50] * 100 + [161, 200] * 6 + [70] * 16, "k", 2064, 1001, 160),
         "long_small": ([64] * 64 + [45] * 63 + [1], "k", 2064, 1024, 160),
         "long_row_major": ([50] * 100 + [161, 200] * 6 + [70] * 16, "nd", 2048, 1008, 160)}


@pytest.mark.parametrize("name", sorted(FORMS))
def test_forms_by_sizes_swiglu_equal_a_forced_height(aclnn, dev, monkeypatch, name):
    sizes, layout, K, columns, want_rows = FORMS[name]
    E, M = len(sizes), sum(sizes)
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.empty((M, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    w = torch.empty((E, 2 * columns, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    view, nz = _weights(w, layout)
    scale, x_scale = torch.rand((E, 2 * columns), device=dev, generator=g) * 1e-3, torch.rand((M,), device=dev, generator=g) * 1e-2
    cumsum = torch.cumsum(torch.tensor(sizes), 0).to(dev)

    def call():
        out = (torch.full((M, columns), 7, dtype=torch.int8, device=dev), torch.full((M,), 7.0, device=dev))
        return aclnn.grouped_matmul_swiglu_quant(x, view, cumsum, scale, x_scale, out=out, weight_nz=nz)

    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    (y, ys), rows = _spanned(aclnn, call)
    assert rows == want_rows
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "96")
    (y96, ys96), rows = _spanned(aclnn, call)
    assert rows == 96 and torch.equal(y, y96) and torch.equal(ys, ys96)


@pytest.mark.parametrize("name,K,N,want_rows", [("dealt", 1280, 2208, 64), ("begun", 1280, 2208, 192), ("some_begun", 1024, 2208, 192), ("long_small", 2064, 2208, 160)])
def test_forms_by_sizes_down(aclnn, monkeypatch, name, K, N, want_rows):
    monkeypatch.delenv("OPAPI_GEMM_TILE_M", raising=False)
    (got, want), rows = _spanned(aclnn, lambda: _run(aclnn, FORMS[name][0], N, K, "k", torch.bfloat16, K))
    assert rows == want_rows
    assert torch.equal(got, want)


# 256-row SwiGLU tiles ask for a tile's scales behind the one before, into two places in turn: three and more tiles a workgroup, of one k-step and
# more, from shares (K below 1024) and drawn
@pytest.mark.parametrize("K", [128, 272, 1024])
def test_scales_of_tiles_in_a_row(aclnn, dev, monkeypatch, K):
    sizes, columns = [300, 256, 0, 299, 301] * 20, 512
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "256")
    got, want = _run(aclnn, sizes, 2 * columns, K, "k", torch.bfloat16, K)
    assert torch.equal(got, want)
    E, M = len(sizes), sum(sizes)
    g = torch.Generator(device=dev).manual_seed(K)
    x = torch.empty((M, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    w = torch.empty((E, 2 * columns, K), dtype=torch.int8, device=dev).random_(-127, 128, generator=g)
    scale, x_scale = torch.rand((E, 2 * columns), device=dev, generator=g) * 1e-3, torch.rand((M + 1,), device=dev, generator=g) * 1e-2
    cumsum = torch.cumsum(torch.tensor(sizes), 0).to(dev)

    def call():
        return aclnn.grouped_matmul_swiglu_quant(x, w.transpose(1, 2), cumsum, scale, x_scale[1:])

    y, ys = call()
    monkeypatch.setenv("OPAPI_GEMM_TILE_M", "96")
    y96, ys96 = call()
    assert torch.equal(y, y96) and torch.equal(ys, ys96)
