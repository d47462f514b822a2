"""Operands whose contiguous extent is no multiple of four floats or that start at an odd float: the
products' moved-back last tiles and shifted K tails (lh_gemm_ws_f32), the vocabulary kernels' guarded
last quad (lh_softmax_fwd_f32, lh_logsoftmax_xent_f32, lh_softmax_xent_grad_f32, lh_beam_topk_f32), and
the reduction of split planes, against float64; and copies of strided blocks.

Tolerances: a product of K terms rounds K + 8 times at most, each by 2^-24 of the sum of magnitudes.
"""
import numpy as np
import pytest
import scipy.special
import torch

from tests.conftest import assert_close

pytestmark = pytest.mark.gpu


def _odd(a, off):
    """a (column-major) on the GPU, `off` floats behind a 16-byte boundary, NaN around it."""
    flat = np.ascontiguousarray(a.T).ravel()
    buf = torch.full((flat.size + 64,), float("nan"), device="cuda")
    view = buf[off: off + flat.size]
    view.copy_(torch.from_numpy(flat))
    return view


# M, N, Ks, transA, transX.  Tails of 1, 2 and 3 past whole slabs of 16 to 128 k, in one segment and in two, with
# either operand or both contiguous along k; tiles moved back along m, along n and along both.
SHAPES = [(33, 5, (4,), False, False), (33, 5, (17,), False, False), (131, 3, (18,), True, False),
          (63, 34, (16,), False, True), (35, 33, (19, 5), False, True), (63, 40, (130,), False, False),
          (129, 97, (67, 18), True, False), (131, 3, (5,), True, False), (257, 129, (33,), False, True),
          (1003, 84, (250, 131), False, False), (31, 30, (9,), False, False), (40, 31, (7,), False, True),
          (34, 34, (3,), True, False), (5001, 12, (256,), False, False), (256, 130, (5001,), True, False),
          (131, 40, (129,), True, False), (70, 45, (130, 67), True, False), (133, 50, (131, 259), False, False),
          (129, 131, (257, 18), False, True), (1001, 1027, (35,), False, True), (130, 70, (66, 129, 5), True, False)]
RAGGED_CONFIGS = {0, 3, 7, 12, 15, 18, 24, 32, 35, 36}


def _kernel(M, N, Ks, tA, tX, off, tile):
    """What takes the product: 'aligned', 'ragged' or 'generic'; tile = (config, BM, BN) or None for any."""
    extents = ([M] if not tA else list(Ks)) + ([N] if tX else list(Ks))
    if off == 0 and all(e % 4 == 0 for e in extents):
        return "aligned"
    ragged_m, ragged_n = not tA and M % 4 != 0, tX and N % 4 != 0
    if (ragged_m and M < 32) or (ragged_n and N < 32) or ((tA or not tX) and min(Ks) < 4):
        return "generic"
    if len(Ks) == 1 and Ks[0] <= 16:
        return "generic"
    if tile is None:
        return "ragged"
    cfg, bm, bn = tile
    return "ragged" if cfg in RAGGED_CONFIGS and not (ragged_m and bm > M) and not (ragged_n and bn > N) else "generic"


@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("M,N,Ks,tA,tX", SHAPES)
def test_ragged_products(lh, M, N, Ks, tA, tX, splits):
    rng = np.random.default_rng(M * 131 + N)
    L = lh.load()
    As = [rng.uniform(-1, 1, (K, M) if tA else (M, K)).astype(np.float32) for K in Ks]
    Xs = [rng.uniform(-1, 1, (N, K) if tX else (K, N)).astype(np.float32) for K in Ks]
    want = np.zeros((M, N))
    mag = np.zeros((M, N))
    for A, X in zip(As, Xs):
        a, x = (A.T if tA else A).astype(np.float64), (X.T if tX else X).astype(np.float64)
        want += a @ x
        mag += np.abs(a) @ np.abs(x)
    C0 = rng.uniform(-1, 1, (M, N)).astype(np.float32)
    bias = rng.uniform(-1, 1, M).astype(np.float32)
    limit = (sum(Ks) + 8) * 2.0 ** -24 * (mag + np.abs(C0) + np.abs(bias[:, None]))
    ws = torch.full((4 << 20,), float("nan"), device="cuda")
    n_cfg = L.lh_gemm_set_config_override(-1)
    ran = set()
    try:
        L.lh_gemm_set_splits_override(splits)
        for cfg in [-1] + list(range(n_cfg)):
            L.lh_gemm_set_config_override(cfg)
            for off in (0, 1, 3):
                segs = [(_odd(A, off), A.shape[0], _odd(X, off), X.shape[0], K)
                        for A, X, K in zip(As, Xs, Ks)]
                name = lh.gemm_kernel_name(M, N, segs, transA=tA, transX=tX, workspace_bytes=16 << 20)
                info = lh.gemm_config_info(cfg, tA, tX) if cfg >= 0 else None
                form = _kernel(M, N, Ks, tA, tX, off, (cfg, info["BM"], info["BN"]) if info else None)
                assert (form == "generic") == name.startswith("gemm_generic_kernel<"), (name, cfg, off)
                assert (form == "ragged") == (name.startswith("gemm_kernel<") and name.count(",") == 8), (name, cfg, off)
                if cfg >= 0 and form != "generic":
                    assert name.startswith("gemm_kernel<%d, %d, %d, %d, %d, %d," % tuple(
                        info[k] for k in ("BM", "BN", "WM", "WN", "WK", "BK"))), (name, cfg)
                    if form == "ragged":
                        ran.add(cfg)
                ldc = M + 3                       # three guard rows behind every column
                out = np.full((ldc, N), 7.0, np.float32)
                out[:M] = C0
                dC = torch.from_numpy(np.ascontiguousarray(out.T).ravel()).cuda()
                lh.gemm(M, N, segs, dC, ldc, transA=tA, transX=tX, beta=0.5,
                        bias=torch.from_numpy(bias).cuda(), workspace=ws)
                got = dC.cpu().numpy().reshape(N, ldc).T
                assert np.all(got[M:] == 7.0), f"config {cfg}: rows behind the result were written"
                err = np.abs(got[:M] - (want + 0.5 * C0 + bias[:, None]))
                assert np.all(err <= limit), f"config {cfg} offset {off}: {err.max()} at {np.argmax(err - limit)}"
    finally:
        L.lh_gemm_set_config_override(-1)
        L.lh_gemm_set_splits_override(0)
    if min(M, N) >= 129 and min(Ks) > 16:     # large enough for every ragged configuration
        assert ran == RAGGED_CONFIGS, ran


# 768 and 1536 rows: the last a short ragged column may have; up to 3072 rows fill fewer wavefronts than there are
# candidates
@pytest.mark.parametrize("V", [13, 501, 767, 769, 1535, 1537, 3001, 3073, 4097, 8191, 30003, 65533])
@pytest.mark.parametrize("off", [0, 1])
def test_ragged_columns(lh, V, off):
    rng = np.random.default_rng(V + off)
    B, K = 7, 13
    z = rng.normal(0, 3, (V, B)).astype(np.float32)
    z[:, 1] = np.round(z[:, 1])              # ties
    z[:, 2] = 0.25                           # everything ties
    z[V - 1, 3] = 40.0                       # the last row of the partial quad wins
    if V > K:
        z[5:, 4] = -np.inf                   # fewer finite rows than candidates
    tgt = rng.integers(0, V, B).astype(np.int32)
    tgt[0], tgt[4] = V - 1, 2
    mask = np.array([1, 1, 0, 1, 1, 1, 1], np.int32)
    dz, dt, dm = _odd(z, off), torch.from_numpy(tgt).cuda(), torch.from_numpy(mask).cuda()
    z64 = z.astype(np.float64)
    logp = z64 - scipy.special.logsumexp(z64, axis=0)
    p = np.exp(logp)

    def fresh():
        return torch.full((V * B + 8,), 7.0, device="cuda")[1:]

    out = fresh()
    lh.softmax_fwd(dz, V, None, V, B, out, V)
    got = out.cpu().numpy()
    assert_close(got[:V * B].reshape(B, V).T, p, "probabilities", rtol=2e-6, atol=1e-9)
    assert np.all(got[V * B:] == 7.0)

    lt, loss = torch.zeros(B, dtype=torch.float64, device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda")
    lh.logsoftmax_xent(dz, V, None, V, B, dt, dm, lt, loss)
    # double exponentials, as in the strided kernel: only the fp32 logits bound the result
    assert_close(lt.cpu().numpy(), logp[tgt, np.arange(B)], "log p", rtol=1e-12, atol=1e-12)
    assert_close(loss.cpu().numpy()[0], (logp[tgt, np.arange(B)] * mask).sum(), "loss", rtol=1e-12, atol=1e-12)

    out = fresh()
    loss.zero_()
    lh.softmax_xent_grad(dz, V, None, V, B, dt, dm, out, V, lt, loss)
    got = out.cpu().numpy()
    onehot = np.zeros((V, B))
    onehot[tgt, np.arange(B)] = 1.0
    assert_close(got[:V * B].reshape(B, V).T, (onehot - p) * mask, "output error", rtol=4e-6, atol=2e-7)
    assert np.all(got[V * B:] == 7.0)

    cl, ci = torch.empty(K * B, device="cuda"), torch.empty(K * B, dtype=torch.int32, device="cuda")
    le = torch.empty(B, device="cuda")
    lh.beam_topk(dz, V, None, V, B, K, 1, cl, ci, le)
    gi, gl = ci.cpu().numpy().reshape(B, K), cl.cpu().numpy().reshape(B, K)
    for b in range(B):
        order = np.lexsort((np.arange(V), -z64[:, b]))[:K]
        assert gi[b].tolist() == order.tolist(), f"column {b}"
        finite = np.isfinite(logp[order, b])
        assert np.array_equal(gl[b][~finite], logp[order, b][~finite])   # -inf
        assert_close(gl[b][finite], logp[order, b][finite], f"column {b} scores", rtol=1e-5, atol=1e-5)
    assert_close(le.cpu().numpy(), logp[1], "log p(<EOF>)", rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("K", [1, 4, 16, 17, 64])
@pytest.mark.parametrize("V", [100, 128, 129, 500, 769, 772, 1088, 1092, 2000, 3073, 3076, 4096, 4100])
def test_candidates_of_short_columns(lh, V, K):
    """Columns that fill few or partly filled groups: nothing of them, all of them or the K best pass the first
    threshold.  Aligned and ragged; ties, one value everywhere, few finite values, winners packed together."""
    rng = np.random.default_rng(V * 100 + K)
    B = 6
    z = rng.normal(0, 3, (V, B)).astype(np.float32)
    z[:, 1] = np.round(z[:, 1])
    z[:, 2] = -1.5
    z[max(1, K - 1):, 3] = -np.inf           # fewer finite rows than candidates
    z[:, 4] = np.sort(z[:, 4])               # the winners in one wavefront, at the end
    z[:, 5] = np.sort(z[:, 5])[::-1]         # ... at the start
    z64 = z.astype(np.float64)
    logp = z64 - scipy.special.logsumexp(z64, axis=0)
    cl, ci = torch.full((K * B,), 7.0, device="cuda"), torch.full((K * B,), -7, dtype=torch.int32, device="cuda")
    le = torch.empty(B, device="cuda")
    for off in (0, 1):
        lh.beam_topk(_odd(z, off), V, None, V, B, K, 1, cl, ci, le)
        gi, gl = ci.cpu().numpy().reshape(B, K), cl.cpu().numpy().reshape(B, K)
        for b in range(B):
            order = np.lexsort((np.arange(V), -z64[:, b]))[:K]
            assert gi[b].tolist() == order.tolist(), f"column {b} offset {off}"
            want = logp[order, b]
            finite = np.isfinite(want)
            assert np.array_equal(gl[b][~finite], want[~finite])
            assert_close(gl[b][finite], want[finite], f"column {b} scores", rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("V", [515, 1027, 2051, 4099])
def test_partial_nan_column(lh, V):
    """A column of NaN holds no candidate: K rounds of arg-max over nothing, as the strided kernel gives."""
    B, K = 2, 5
    z = np.full((V, B), np.nan, np.float32)
    z[:, 1] = np.arange(V) / V
    cl, ci = torch.zeros(K * B, device="cuda"), torch.zeros(K * B, dtype=torch.int32, device="cuda")
    le = torch.empty(B, device="cuda")
    lh.beam_topk(_odd(z, 0), V, None, V, B, K, 1, cl, ci, le)
    gi = ci.cpu().numpy().reshape(B, K)
    assert gi[0].tolist() == [0x7fffffff] * K
    assert gi[1].tolist() == [V - 1 - i for i in range(K)]


@pytest.mark.parametrize("rows,cols,ld_dst,ld_src", [(4, 1, 4, 16), (1000, 7, 1000, 4000), (37, 5, 37, 148),
                                                     (8, 3, 9, 32), (1, 300, 1, 4)])
@pytest.mark.parametrize("off", [0, 1])
def test_copy_block(lh, rows, cols, ld_dst, ld_src, off):
    """lh_copy_block_f32: exact, and nothing beside the block is written."""
    rng = np.random.default_rng(rows)
    src = torch.from_numpy(rng.random(ld_src * cols + off + 8, dtype=np.float32)).cuda()
    dst = torch.full((ld_dst * cols + off + 8,), 7.0, device="cuda")
    lh.check(lh.load().lh_copy_block_f32(dst[off:].data_ptr(), ld_dst, src[off:].data_ptr(), ld_src, rows, cols,
                                         torch.cuda.current_stream().cuda_stream), "lh_copy_block_f32")
    want = np.full(ld_dst * cols + off + 8, 7.0, np.float32)
    s = src.cpu().numpy()
    for c in range(cols):
        want[off + c * ld_dst: off + c * ld_dst + rows] = s[off + c * ld_src: off + c * ld_src + rows]
    assert np.array_equal(dst.cpu().numpy(), want)


@pytest.mark.parametrize("H,D,W", [(64, 10, 21), (1500, 3, 7), (100, -1, 40), (68, 20, 41)])
def test_padded_columns_read_no_column_of_their_own(lh, H, D, W):
    """A column with mask 0, or whose window lies outside the caller's steps, may carry any hs_col entry: it
    reads nothing through it.  NaN behind every column that is not such a column's neighbour shows a use."""
    rng = np.random.default_rng(H)
    S, B = 40, 4
    hs = rng.normal(0, 1, (S, 2, H)).astype(np.float32)      # two columns of states
    wa, t1, vp = (rng.normal(0, 0.1, n).astype(np.float32) for n in ((B, H), (B, H), H))
    hs_col = np.array([1, 1 << 20, 0, 1 << 20], np.int32)     # columns 1 and 3 point nowhere
    info = np.array([S, S, S, S, 0, 0, 0, 5 * S], np.int32)   # lengths, offsets: column 3 lies past the steps
    mask = np.array([1, 0, 1, 1], np.int32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    f = lambda n: torch.full((n,), float("nan"), device="cuda")     # noqa: E731
    p, sg, al, ce, ctx = f(B), f(B), f(B * W), f(B * W), f(B * H)
    idx = torch.zeros(B * W, dtype=torch.int32, device="cuda")
    lh.attn_core_fwd(H, B, D, W, S, d(t1), d(vp), d(wa), d(hs), 2 * H, H, d(hs_col), d(info), d(mask), p, sg, idx, al,
                     ce, ctx)
    got, w, at = ctx.cpu().numpy().reshape(B, H), al.cpu().numpy().reshape(W, B), idx.cpu().numpy().reshape(W, B)
    assert np.all(got[1] == 0) and np.all(got[3] == 0) and np.all(at[:, 1] == -1)
    for b in (0, 2):
        want = sum(w[j, b].astype(np.float64) * hs[S - 1 - at[j, b], hs_col[b]] for j in range(W) if at[j, b] >= 0)
        assert np.abs(got[b] - want).max() <= 2.0 ** -22 * W * np.abs(hs).max()
