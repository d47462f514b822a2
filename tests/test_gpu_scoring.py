"""Scoring of whole minibatches (lnmt_get_error): the output projection and the loss run over groups of steps.
Several groups and an uneven last one, groups of one step in the model's own buffers, a training model's
buffers, split products, an empty target.

Tolerance of a log-probability: its logits carry H + 8 roundings of 2^-24 of the sum of magnitudes each (twice:
the word's and the normaliser's), the normaliser's exponentials a relative 2^-20 (exponents up to 20 through
one multiplication and v_exp_f32)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def host():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from linmt_amd import host as h
    h.load()
    return h


def _language_model(host, rng, H, V, B, T, **kw):
    m = host.Model(1, H, V, V, longest_sentence=T, attention_mode=0, feed_input=False, minibatch_size=B,
                   sequence_to_sequence=False, **kw)
    u = lambda *s: rng.uniform(-0.3, 0.3, s).astype(np.float32)  # noqa: E731
    P = {"tgt.0.W": u(H, V), "softmax.D": u(V, H), "softmax.b_d": u(V)}
    for g in "ifco":
        P.update({f"tgt.0.W_h{g}": u(H, H), f"tgt.0.M_{g}": u(H, H), f"tgt.0.b_{g}": u(H)})
    m.set_params(P)
    lengths = rng.integers(1, T + 1, B)
    lengths[0] = T
    tin, tout = (rng.integers(0, V, (B, T)).astype(np.int32) for _ in range(2))
    pad = np.arange(T)[None, :] >= lengths[:, None]
    tin[pad], tout[pad] = -1, -1
    return m, P, tin, tout


def _expected(m, P, tout, H, B):
    """Per-column sums of log p(target) from the model's states, in float64, and their error bounds."""
    D, b = P["softmax.D"].astype(np.float64), P["softmax.b_d"].astype(np.float64)
    want, bound = np.zeros(B), np.zeros(B)
    for t in range(tout.shape[1]):
        h = m.get_state(0, 1, 0, t, H, B).astype(np.float64)
        for c0 in range(0, B, 256):
            cols = np.flatnonzero(tout[c0:c0 + 256, t] >= 0) + c0
            if not len(cols):
                continue
            z = D @ h[:, cols] + b[:, None]
            top = z.max(axis=0)
            want[cols] += z[tout[cols, t], np.arange(len(cols))] - top - np.log(np.exp(z - top).sum(axis=0))
            mag = (np.abs(D).max(axis=0) @ np.abs(h[:, cols])) + np.abs(b).max()
            bound[cols] += 2 * (H + 8) * 2.0 ** -24 * mag + 2.0 ** -20
    return want, bound


# the limit of a group is 2^27 logits: all steps at once, 14 + 14 + 13 steps, three times one step
@pytest.mark.parametrize("H,V,B,T,groups", [(32, 5003, 9, 10, 1), (64, 30000, 256, 41, 3), (16, 66000, 1024, 3, 3)])
def test_groups_of_steps(host, H, V, B, T, groups):
    m, P, tin, tout = _language_model(host, np.random.default_rng(T), H, V, B, T)
    m.profile(2)
    got = m.get_error(None, tin, tout, None)
    totals = m.profile_totals()
    assert sum(v["launches"] for k, v in totals.items() if k.startswith("logits_gemm")) == groups, totals.keys()
    want, bound = _expected(m, P, tout, H, B)
    assert abs(got - want.sum()) <= bound.sum(), (got, want.sum(), bound.sum())
    # fewer columns than the model has: a step at a time
    part = m.get_error(None, tin[:B - 1], tout[:B - 1], None)
    assert abs(part - want[:B - 1].sum()) <= bound.sum(), (part, want[:B - 1].sum())
    m.close()


def test_training_model_scores_in_its_own_buffers(host):
    H, V, B, T = 64, 30000, 64, 40
    m, P, tin, tout = _language_model(host, np.random.default_rng(1), H, V, B, T, training=dict(grad_clip_mode=0))
    words = np.unique(tin[tin >= 0]).astype(np.int32)
    trained = m.compute_gradients(None, tin, tout, None, None, words)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    got = m.get_error(None, tin, tout, None)
    assert free - torch.cuda.mem_get_info()[0] < 32 << 20      # 300 MB of logits, in place
    want, bound = _expected(m, P, tout, H, B)
    assert abs(got - want.sum()) <= bound.sum() and abs(trained - want.sum()) <= bound.sum()
    m.close()


def test_grouping_does_not_switch_scoring_to_split_products(host):
    """A step's output projection (64 columns) stays an fp32 product with split products on, so the projection
    of many steps does; nothing else of this minibatch is large enough for them."""
    H, V, B, T = 1024, 16000, 64, 20
    m, P, tin, tout = _language_model(host, np.random.default_rng(2), H, V, B, T, training=dict(grad_clip_mode=0))
    want = m.get_error(None, tin, tout, None)
    m.set_split_products(True)
    assert m.get_error(None, tin, tout, None) == want
    m.close()


def test_empty_target(host):
    m, P, tin, tout = _language_model(host, np.random.default_rng(3), 16, 20, 4, 1)
    assert m.get_error(None, tin[:, :0], tout[:, :0], None) == 0.0
    assert m.get_error(None, tin, tout, None) < 0.0
    m.close()
