"""Attention kernels that split a column over wavefronts and groups of threads, at the sizes where the split
changes: slots without a state beside live ones in every group, rows that fill one group, several or more than one
round, and the column counts at which a column gets fewer wavefronts."""
import numpy as np
import pytest
import torch

from conftest import assert_close
from test_gpu_train_kernels import dev, host, uni

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,B,S,D", [(36, 6, 40, 10), (510, 5, 30, 10), (516, 5, 30, 3), (1003, 4, 12, 10),
                                     (2048, 5, 30, 10), (4200, 3, 9, 2), (1000, 4, 70, -1), (40, 3, 300, 255),
                                     (36, 257, 300, 255), (64, 256, 20, 4), (64, 257, 20, 4), (1000, 300, 9, 3)])
def test_backward_slots_without_a_state(lh, orc, H, B, S, D):
    """Sentences shorter than the window and columns without a word: slot j of one group is live while slots of
    the others are not.  Rows of dhs that no slot points at keep their bits.  Sixteen wavefronts a column up to
    256 columns with more than 8 slots, else eight."""
    rng = np.random.default_rng(H + S)
    lens = rng.integers(1, S + 1, size=B)
    lens[:3] = S, 1, 2
    bi = np.concatenate([lens, S - lens]).astype(np.int32)
    mask = np.ones(B, np.int32)
    mask[-1] = 0
    hs, dhs0 = uni(rng, S * B * H, s=0.5), uni(rng, S * B * H, s=0.1)
    tanh1, v_p, wa, dctx = np.tanh(uni(rng, H, B)), uni(rng, H, s=0.05), uni(rng, H, B, s=0.1), uni(rng, H, B, s=0.1)
    fwd = orc.attn_core_fwd(H, B, D, S, S, tanh1, v_p, wa, hs, B * H, H, None, bi, mask)
    want = orc.attn_core_bwd(H, B, D, S, S, dctx, tanh1, v_p, wa, hs, B * H, H, bi, fwd, dhs0)
    got = []
    for _ in range(2):
        dhs = dev(dhs0)
        hsum, u, w = (torch.full((H * B,), float("nan"), device="cuda") for _ in range(3))
        lh.attn_core_bwd(H, B, D, S, S, dev(dctx), dev(tanh1), dev(v_p), dev(wa), dev(hs), B * H, H, dev(bi),
                         dev(fwd["p_t"]), dev(fwd["sigma"]), dev(fwd["indices"]), dev(fwd["align"]),
                         dev(fwd["cached_exp"]), dhs, hsum, u, w)
        got.append((host(hsum, (H, B)), host(dhs, (S * B * H,)).reshape(S, B, H), host(u, (H, B)), host(w, (H, B))))
    assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(*got))
    assert_close(got[0][0], want["hsum"], "hsum", atol=2e-5)
    assert_close(got[0][1].ravel(), np.ravel(want["dhs"]), "dhs", atol=2e-5)
    if D >= 0:
        assert_close(got[0][2], want["u"], "u", atol=2e-5)
        assert_close(got[0][3], want["w"], "w", atol=2e-5)
    for b in range(B):
        index = fwd["indices"][b]
        tau = S - 1 - index[index >= 0]      # left-padded: timestep of source position i
        idle = np.setdiff1d(np.arange(S), tau)
        assert np.array_equal(got[0][1][idle, b], dhs0.reshape(S, B, H)[idle, b])


@pytest.mark.parametrize("H,D,S", [(64, 20, 50), (38, -1, 30), (132, 130, 300), (512, -1, 60)])
@pytest.mark.parametrize("B", [512, 513, 1024, 1025, 2048, 2049])
def test_forward_at_the_column_counts_of_the_split(lh, orc, H, D, S, B):
    """A column has 16 wavefronts up to 512 columns, 8 up to 1024 and past 2048 (or for windows of more than 256
    slots), 4 between.  Against the oracle; and what does not depend on the split (position, window, weights)
    has the bits it has among 512 columns."""
    rng = np.random.default_rng(H + B)
    W, cols = 2 * D + 1 if D >= 0 else S, 40
    hs, v_p = uni(rng, S * cols * H, s=0.5), uni(rng, H, s=0.1)
    tanh1, wa = np.tanh(uni(rng, H, B)), uni(rng, H, B, s=0.1)
    lens = rng.integers(1, S + 1, size=B)
    lens[:2], lens[-1] = (S, 1), S
    bi, mask = np.concatenate([lens, S - lens]).astype(np.int32), (rng.random(B) < 0.9).astype(np.int32)
    mask[0] = mask[-1] = 1
    hs_col = rng.integers(0, cols, B).astype(np.int32)

    def run(n):
        f = lambda k: torch.full((k,), float("nan"), device="cuda")  # noqa: E731
        p, sg, al, ce, ctx = f(n), f(n), f(n * W), f(n * W), f(n * H)
        ix, vt = (torch.zeros(k, dtype=torch.int32, device="cuda") for k in (n * W, n))
        lh.attn_core_fwd(H, n, D, S, S, dev(tanh1[:, :n]), dev(v_p), dev(wa[:, :n]), dev(hs), cols * H, H, dev(hs_col[:n]),
                         dev(np.concatenate([bi[:n], bi[B:B + n]])), dev(mask[:n]), p, sg, ix, al, ce, ctx, vt)
        return dict(p_t=host(p, (n,)), indices=host(ix, (n, W)), align=host(al, (n, W)), viterbi=host(vt, (n,)),
                    ctx=host(ctx, (H, n)))

    got, few = run(B), run(512)
    want = orc.attn_core_fwd(H, B, D, S, S, tanh1, v_p, wa, hs, cols * H, H, hs_col, bi, mask)
    assert np.array_equal(got["indices"], want["indices"])
    for name in ("align", "ctx") + (("p_t",) if D >= 0 else ()):
        assert_close(got[name], want[name], name)
    for name in ("p_t", "indices", "align", "viterbi"):
        assert np.array_equal(got[name][:512], few[name], equal_nan=True), name
