"""Operands whose contiguous extent is no multiple of four floats or that start at an odd float: the
products' moved-back last tiles and shifted K tails (lh_gemm_ws_f32), the vocabulary kernels' guarded
last quad (lh_softmax_fwd_f32, lh_logsoftmax_xent_f32, lh_softmax_xent_grad_f32, lh_beam_topk_f32), and
the reduction of split planes, against float64.

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


# M, N, Ks, transA, transX
SHAPES = [(33, 5, (4,), False, False), (35, 33, (19, 5), False, True), (63, 40, (130,), False, False),
          (129, 97, (67, 18), True, False), (131, 3, (5,), True, False), (257, 129, (33,), False, True),
          (1003, 84, (250, 131), False, False), (31, 30, (9,), False, False), (40, 31, (7,), False, True),
          (34, 34, (3,), True, False), (5001, 12, (256,), False, False), (256, 130, (5001,), True, False)]


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
    names = set()
    try:
        L.lh_gemm_set_splits_override(splits)
        for cfg in [-1] + list(range(n_cfg)):
            L.lh_gemm_set_config_override(cfg)
            for off in (0, 1, 3):
                segs = [(_odd(A, off), A.shape[0], _odd(X, off), X.shape[0], K)
                        for A, X, K in zip(As, Xs, Ks)]
                if cfg < 0:
                    names.add(lh.gemm_kernel_name(M, N, segs, transA=tA, transX=tX, workspace_bytes=16 << 20))
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
    generic = (not tA and M % 4 and M < 32) or (tX and N % 4 and N < 32) or ((tA or not tX) and min(Ks) < 4)
    assert all(n.startswith("gemm_generic" if generic else "gemm_kernel") for n in names), names
