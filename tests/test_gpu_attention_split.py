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
                                     (2048, 5, 30, 10), (4200, 3, 9, 2), (1000, 4, 70, -1)])
def test_backward_slots_without_a_state(lh, orc, H, B, S, D):
    """Sentences shorter than the window and columns without a word: slot j of one group is live while slots of
    the others are not.  Rows of dhs that no slot points at keep their bits."""
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
