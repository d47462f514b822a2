"""Products on the streamed tiles (eight wavefronts, a 32x32 block each, operands loaded straight into LDS)
against float64: the edges of tiles and slabs, segments that end inside a slab or within a wavefront's share of
one, segments of unlike leading dimensions, K split over workgroups."""
import pytest

pytestmark = pytest.mark.gpu

CONFIGS = [13, 14, 15, 19]


@pytest.fixture()
def lh():
    from linmt_amd import lib
    lib.load()
    yield lib
    lib.load().lh_gemm_set_config_override(-1)
    lib.load().lh_gemm_set_splits_override(0)


def operand(torch, rows, cols, pad, seed):
    """rows x cols column-major with leading dimension rows + pad; what lies between is NaN: never to be used."""
    g = torch.Generator("cuda").manual_seed(seed)
    full = torch.full((cols, rows + pad), float("nan"), device="cuda")
    full[:, :rows] = torch.randn(cols, rows, device="cuda", generator=g)
    return full, full[:, :rows].T.double()


@pytest.mark.parametrize("tA", [False, True], ids=["NN", "TN"])
@pytest.mark.parametrize("M,N,Ks,splits", [
    (20, 12, (260,), 1), (256, 24, (1024, 28), 1), (100, 33, (512, 36, 292), 1), (996, 64, (1000,), 1),
    (1000, 128, (1000, 4), 1), (200, 36, (1000,), 2)])
def test_narrow_product_matches_float64(lh, tA, M, N, Ks, splits):
    """Tiles of 16 rows and 16 or 32 columns, which no override names: chosen at these sizes."""
    import torch
    lh.load().lh_gemm_set_splits_override(splits)
    any_matrix = torch.empty(max(M, N) * 2048, device="cuda")
    segs = [(any_matrix, 2048, any_matrix, 2048, K) for K in Ks]
    name = lh.gemm_kernel_name(M, N, segs, tA, False, 64 * M * N)
    assert name.startswith("gemm_kernel<16, %d," % (32 if N == 128 else 16)), name
    test_streamed_product_matches_float64(lh, -1, tA, False, M, N, Ks, splits)


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("tA,tX", [(False, False), (True, False), (False, True)], ids=["NN", "TN", "NT"])
@pytest.mark.parametrize("M,N,Ks,splits", [
    (4, 4, (4,), 1),              # one unit of everything
    (32, 32, (8,), 1),            # less than a wavefront's share of a slab
    (36, 20, (64,), 1),           # one row unit past a tile, one slab of the shallow tiles
    (64, 64, (132, 20), 1),       # a segment that ends in the first wavefront's share, then a short one
    (100, 68, (16, 512, 60), 1),  # four slabs in flight and the ring round more than once
    (1000, 64, (1000, 1000), 1),
    (200, 36, (1000,), 4),        # K split over workgroups
    (200, 36, (260, 20), 2),
])
def test_streamed_product_matches_float64(lh, config, tA, tX, M, N, Ks, splits):
    import torch
    segs, want, bound = [], 0, 0
    for i, K in enumerate(Ks):
        pad = 4 * (i + 1)
        a, a64 = operand(torch, K if tA else M, M if tA else K, pad, 10 * i)
        x, x64 = operand(torch, N if tX else K, K if tX else N, pad + 4, 10 * i + 1)
        a64, x64 = (a64.T if tA else a64), (x64.T if tX else x64)
        segs.append((a, a.shape[1], x, x.shape[1], K))
        want = want + a64 @ x64
        bound = bound + a64.abs() @ x64.abs()
    bias = torch.randn(M, device="cuda")
    old = torch.randn(N, M, device="cuda")
    out = old.clone()
    ws = torch.empty(16 * M * N, device="cuda")
    lib = lh.load()
    lib.lh_gemm_set_config_override(config)
    lib.lh_gemm_set_splits_override(splits)
    lh.gemm(M, N, segs, out, M, transA=tA, transX=tX, beta=1.0, bias=bias, workspace=ws)
    torch.cuda.synchronize()
    want = want + old.T.double() + bias.double()[:, None]
    # K products and their sum in fp32, in any order, plus the two addends: (K + 3) roundings of the sum of
    # magnitudes at most
    bound = (sum(Ks) + 3) * 2.0 ** -24 * (bound + old.T.double().abs() + bias.double().abs()[:, None])
    assert bool(((out.T.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("form", [0, 1], ids=["16x16", "16x32"])
@pytest.mark.parametrize("tA,M,N,Ks,splits", [
    (False, 4, 1, (4,), 1), (False, 20, 33, (32,), 1), (False, 100, 17, (288, 4), 1), (False, 64, 48, (1028, 12), 3),
    (True, 1, 1, (4,), 1), (True, 17, 33, (36,), 1), (True, 101, 16, (260, 8, 1000), 1), (True, 33, 31, (1028,), 4),
    (True, 1003, 5, (516, 4), 2)])
def test_narrow_tiles_by_name(lh, form, tA, M, N, Ks, splits):
    """The tiles of 16 rows at the edges of tiles, slabs and shares, whatever the cost model would take there; a
    transposed A may have any number of rows."""
    import torch
    lib = lh.load()
    config = lib.lh_gemm_set_config_override(-1) + form
    lib.lh_gemm_set_config_override(config)
    any_matrix = torch.empty(16, device="cuda")
    info = lh.gemm_config_info(config, tA, False)
    assert (info["BM"], info["BN"]) == (16, 16 * (form + 1)) and info["occupancy"] >= 1
    name = lh.gemm_kernel_name(M, N, [(any_matrix, 2048, any_matrix, 2048, K) for K in Ks], tA, False, 64 * M * N)
    assert name.startswith("gemm_kernel<16, %d," % (16 * (form + 1))), name
    test_streamed_product_matches_float64(lh, config, tA, False, M, N, Ks, splits)


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("M,N,Ks,splits", [
    (32, 32, (1,), 1), (36, 32, (7,), 1), (64, 36, (66, 3), 1), (100, 68, (131, 1, 513), 1), (200, 36, (1001,), 3)])
def test_streamed_product_over_any_k(lh, config, M, N, Ks, splits):
    """X transposed (weight gradients): both operands are contiguous along the columns, and K may be any number."""
    import torch
    lh.load().lh_gemm_set_config_override(config)
    any_matrix = torch.empty(16, device="cuda")
    name = lh.gemm_kernel_name(M, N, [(any_matrix, 2048, any_matrix, 2048, K) for K in Ks], False, True, 64 * M * N)
    assert name.startswith("gemm_kernel<") and name.count(",") == 7, name
    test_streamed_product_matches_float64(lh, config, False, True, M, N, Ks, splits)


def test_narrow_tiles_named_where_they_cannot_run(lh):
    """No such tile for a transposed X: the override falls back like any other that does not fit, and there is no
    configuration behind the two."""
    import torch
    lib = lh.load()
    n = lib.lh_gemm_set_config_override(-1)
    with pytest.raises(lh.LinmtHipError):
        lh.gemm_config_info(n, False, True)
    with pytest.raises(lh.LinmtHipError):
        lh.gemm_config_info(n + 2)
    with pytest.raises(lh.LinmtHipError):
        lh.check(min(0, lib.lh_gemm_set_config_override(n + 2)), "override")
    test_streamed_product_matches_float64(lh, n, False, True, 36, 20, (64,), 1)
