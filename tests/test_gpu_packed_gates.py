"""Gate products on packed gate matrices: the layout of lh_gate_pack_f32, the product with its cell
against float64 and against the kernel on the stored matrix, and a model whose weights change
between two passes."""
import numpy as np
import pytest

from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

CONFIGS = [-1, 13, 14, 15, 19]


@pytest.fixture()
def lh():
    from linmt_amd import lib
    lib.load()
    yield lib
    lib.load().lh_gemm_set_config_override(-1)


def _packed(lh, torch, H, W, Ks):
    P = [torch.full((lh.gate_pack_floats(H, K),), float("nan"), device="cuda") for K in Ks]
    lh.gate_pack(H, [(w, w.shape[1], K, p) for w, K, p in zip(W, Ks, P)])
    return P


@pytest.mark.parametrize("H,Ks", [(4, (4,)), (8, (20,)), (36, (36, 12)), (100, (100, 8, 4)), (1000, (1000, 1000))])
def test_pack_layout(lh, H, Ks):
    import torch
    W = [torch.randn(K, 4 * H + 4, device="cuda") for K in Ks]  # column-major, ld = 4H + 4
    for w, K, p in zip(W, Ks, _packed(lh, torch, H, W, Ks)):
        blocks = (H + 7) // 8
        cells = torch.zeros(K, 4, blocks * 8, device="cuda")
        cells[:, :, :H] = w[:, :4 * H].view(K, 4, H)
        want = cells.view(K, 4, blocks, 8).permute(2, 0, 3, 1)
        assert torch.equal(want.flatten(), p)


@pytest.mark.parametrize("H,B,Ks,columns", [
    (256, 16, (260,), 16), (256, 17, (292, 8), 16), (100, 32, (100, 36, 1028), 16), (1000, 1, (1000, 1000), 16),
    (1000, 25, (1000,), 32), (996, 32, (520, 28), 32), (512, 64, (512,), 32)])
def test_narrow_gate_product_with_cell(lh, H, B, Ks, columns):
    """The forms of 16 rows and 16 or 32 columns: remainders of the wavefronts' 32 k, of a slab of 256, of the
    four cells and of the columns; more slabs than the ring holds."""
    import torch
    any_matrix = torch.empty(4 * H * max(Ks), device="cuda")
    name = lh.gate_gemm_lstm_cell_packed_plan(H, B, [(any_matrix, 4 * H, any_matrix, K, K) for K in Ks], True)[1]
    assert name == f"gate_gemm_narrow_kernel<{columns // 16}>"
    test_packed_gate_product_with_cell(lh, -1, H, B, Ks)


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("H,B,Ks", [(4, 1, (4,)), (36, 33, (36,)), (64, 32, (132, 20)), (100, 65, (16, 100, 60)),
                                    (1000, 12, (1000, 1000))])
def test_packed_gate_product_with_cell(lh, config, H, B, Ks):
    """With an addend by column, gate values and the dropped copy kept."""
    import torch
    torch.manual_seed(H + B)
    dev = dict(device="cuda")
    W = [torch.randn(K, 4 * H, **dev) / K ** 0.5 for K in Ks]
    X = [torch.randn(B, K, **dev) for K in Ks]
    table, col = torch.randn(7, 4 * H, **dev), torch.randint(0, 7, (B,), dtype=torch.int32, **dev)
    bias, c_prev, drop = torch.randn(4 * H, **dev), torch.randn(B, H, **dev), torch.rand(B, H, **dev)
    mask = (torch.rand(B, **dev) > 0.2).int()
    pre = sum(x.double() @ w.double() for w, x in zip(W, X)) + table.double()[col.long()] + bias.double()
    i, f, g, o = pre.view(B, 4, H).unbind(1)
    i, f, g, o = torch.sigmoid(i), torch.sigmoid(f), torch.tanh(g), torch.sigmoid(o)
    c = (f * c_prev.double() + i * g)
    h = (o * torch.tanh(c)) * mask[:, None]
    c = c * mask[:, None]
    segs = [(p, 32, x, K, K) for p, x, K in zip(_packed(lh, torch, H, W, Ks), X, Ks)]
    got_c, got_h, got_d = (torch.full((B, H), float("nan"), **dev) for _ in range(3))
    gates = torch.full((B, 4 * H), float("nan"), **dev)
    lh.load().lh_gemm_set_config_override(config)
    lh.gate_gemm_lstm_cell_packed(H, B, segs, bias, c_prev, mask, got_c, got_h, addend=table, ld_addend=4 * H,
                                  addend_col=col, addend_ncols=7, gates=gates, next_drop_mask=drop, keep=0.8,
                                  h_drop=got_d)
    torch.cuda.synchronize()
    # a pre-activation rounds K + 3 times, by 2^-24 of the sum of magnitudes; the cell's derivatives are below 1 in
    # i, f, o (times |c_prev| or 1) and g, and its own functions round a few times more
    mags = sum(x.abs().double() @ w.abs().double() for w, x in zip(W, X)) + table.abs().max() + bias.abs().max()
    tol = ((sum(Ks) + 3) * 2.0 ** -24 * mags.max().item() + 1e-6) * (1 + c_prev.abs().max().item())
    for name, got, want in (("c", got_c, c), ("h", got_h, h), ("gates", gates, torch.cat([i, f, g, o], 1)),
                            ("h_drop", got_d, (drop < 0.8).double() / 0.8 * h)):
        assert (got.double() - want).abs().max().item() <= tol, name


@pytest.mark.parametrize("B", [3, 64])
def test_weights_set_between_passes_reach_the_packed_copy(lh, B):
    """A model that has packed its gates must pack them anew when a matrix is set and after an update."""
    import torch
    from linmt_amd import host
    rng = np.random.default_rng(B)
    H, V, S = 256, 50, 6
    any_matrix = torch.empty(4 * H * H, device="cuda")
    assert lh.gate_gemm_lstm_cell_packed_plan(H, B, [(any_matrix, 4 * H, any_matrix, H, H)] * 2)[0]
    kw = dict(longest_sentence=S + 4, attention_mode=0, minibatch_size=B)
    u = lambda *s: rng.uniform(-0.3, 0.3, size=s).astype(np.float32)  # noqa: E731
    P = {"softmax.D": u(V, H), "softmax.b_d": u(V)}
    for side in ("src", "tgt"):
        P[side + ".0.W"] = u(H, V)
        for layer in range(2):
            for g in "ifco":
                P[f"{side}.{layer}.W_h{g}"], P[f"{side}.{layer}.M_{g}"], P[f"{side}.{layer}.b_{g}"] = u(H, H), u(H, H), u(H)
    src, ti, to = (rng.integers(0, V, (B, S)).astype(np.int32) for _ in range(3))
    info = np.concatenate([np.full(B, S), np.zeros(B)]).astype(np.int32)
    unique = [np.unique(a).astype(np.int32) for a in (src, ti)]
    m = host.Model(2, H, V, V, training=dict(learning_rate=0.5, grad_clip_mode=0), **kw)
    m.set_params(P)
    first = m.compute_gradients(src, ti, to, info, *unique)
    m.update_weights()
    P["src.1.W_hf"] = u(H, H)
    m.set_params({"src.1.W_hf": P["src.1.W_hf"]})
    second = m.compute_gradients(src, ti, to, info, *unique)
    fresh = host.Model(2, H, V, V, **kw)
    shapes = {n: a.shape for n, a in P.items()}
    fresh.set_params({n: np.asfortranarray(m.get_param(n, s)) for n, s in shapes.items()})
    want = fresh.get_error(src, ti, to, info)
    assert abs(first - second) > 1e-2
    assert_close(second, want, "loss with the weights as they are now", rtol=1e-6, atol=1e-4)
    m.close(), fresh.close()


def _training_model(host, rng, H, V, B, longest, layers=2):
    m = host.Model(layers, H, V, V, longest_sentence=longest, attention_mode=0, minibatch_size=B,
                   training=dict(learning_rate=0.1, grad_clip_mode=0))
    u = lambda *s: rng.uniform(-0.1, 0.1, size=s).astype(np.float32)  # noqa: E731
    P = {"softmax.D": u(V, H), "softmax.b_d": u(V)}
    for side in ("src", "tgt"):
        P[side + ".0.W"] = u(H, V)
        for layer in range(layers):
            for g in "ifco":
                P[f"{side}.{layer}.W_h{g}"], P[f"{side}.{layer}.M_{g}"], P[f"{side}.{layer}.b_{g}"] = u(H, H), u(H, H), u(H)
    m.set_params(P)
    return m


def test_training_packs_where_the_pass_is_long_enough(lh):
    """The weights are packed anew for every minibatch: one step does not save what that costs, 24 do."""
    from linmt_amd import host
    rng = np.random.default_rng(5)
    H, V, B = 512, 60, 32
    m = _training_model(host, rng, H, V, B, 28)
    for steps, packed in ((1, False), (24, True)):
        src, ti, to = (rng.integers(0, V, (B, steps)).astype(np.int32) for _ in range(3))
        info = np.concatenate([np.full(B, steps), np.zeros(B)]).astype(np.int32)
        m.profile(2)
        m.compute_gradients(src, ti, to, info, *(np.unique(a).astype(np.int32) for a in (src, ti)))
        names = list(m.profile_totals())
        m.profile(0)
        m.update_weights()
        assert any("gate_gemm_packed_kernel" in n or "gate_gemm_narrow_kernel" in n for n in names) == packed, (steps, names)
    m.close()


def test_without_packed_copies_the_stored_matrices_are_used(lh):
    """What a layer does where the card has no memory to spare: the same results to the rounding of the sums, and copies
    made before are not used."""
    from linmt_amd import host
    rng = np.random.default_rng(9)
    H, V, B, steps = 512, 60, 32, 24
    src, ti, to = (rng.integers(0, V, (B, steps)).astype(np.int32) for _ in range(3))
    info = np.concatenate([np.full(B, steps), np.zeros(B)]).astype(np.int32)
    unique = [np.unique(a).astype(np.int32) for a in (src, ti)]
    m = _training_model(host, rng, H, V, B, 28)
    watched = {n: (H, H) for n in ("src.0.W_hf", "src.1.M_i", "tgt.1.W_ho", "tgt.1.M_c")}
    results = []
    try:
        for off in (0, 1, 0):
            host.set_debug_option("no_packed_gates", off)
            m.profile(2)
            loss = m.compute_gradients(src, ti, to, info, *unique)
            packed = any("gate_gemm_packed_kernel" in n or "gate_gemm_narrow_kernel" in n for n in m.profile_totals())
            m.profile(0)
            assert packed == (off == 0)
            # (gradients add up until the next update)
            results.append((loss, {n: m.get_grad(n, s) / (len(results) + 1) for n, s in watched.items()}))
    finally:
        host.set_debug_option("no_packed_gates", 0)
    for loss, grads in results[1:]:
        assert_close(loss, results[0][0], "loss", rtol=1e-6, atol=1e-4)
        for n in watched:
            # (2-norm; products whose sums are cut at other places give up to 1e-5 in a gradient of this size)
            assert np.linalg.norm(grads[n] - results[0][1][n]) <= 4e-5 * np.linalg.norm(results[0][1][n]), n
    m.close()


@pytest.mark.parametrize("config", [-1, 13, 14, 15, 19, 45, 46])  # 45 and 46: the narrow forms
@pytest.mark.parametrize("f64,clip,addend,kept", [
    (False, 0.0, None, False), (True, 0.0, "column", False),  # scoring without feed input; a decoding step with it
    (True, 0.3, "dense", True), (False, 0.3, "dense", False), (True, 0.0, None, True), (False, 0.0, "column", True)])
@pytest.mark.parametrize("H,B,Ks", [(36, 33, (36,)), (100, 12, (100, 260))])
def test_packed_cell_forms(lh, orc, config, f64, clip, addend, kept, H, B, Ks):
    """Every argument that changes the cell or what it leaves: double sigmoids, columns that take the fp32 ones all the
    same (mask 3: the first step of a streamed sentence), clipping, an addend per column, through a column index or none,
    gate values and the dropped copy kept or not, the cell state in place."""
    import torch
    n = lh.load().lh_gemm_set_config_override(-1)
    assert n == 45
    rng = np.random.default_rng(H + B + 2 * int(f64) + int(kept))
    uni = lambda *s: rng.uniform(-1, 1, s).astype(np.float32)  # noqa: E731
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    W, X = [uni(K, 4 * H) * np.float32(0.3) for K in Ks], [uni(B, K) for K in Ks]  # column-major 4H x K and K x B
    table, col = uni(7, 4 * H), rng.integers(0, 7, B).astype(np.int32)
    bias, c_prev, drop = uni(4 * H), uni(B, H), rng.random((B, H)).astype(np.float32)
    mask = rng.choice(np.array([0, 1, 3], np.int32), B)
    add = {None: None, "column": table[col], "dense": uni(B, 4 * H)}[addend]
    pre = sum(x.astype(np.float64) @ w for x, w in zip(X, W)) + (0 if add is None else add)
    want = [orc.lstm_cell_fwd(pre.T.astype(np.float32), bias, c_prev.T, mask & 1, feed=form, cell_clip=clip)
            for form in (False, f64)]
    gates_want, c_want, h_want = (np.where(mask >= 2, a, b).T for a, b in zip(*want))  # per column
    segs = [(p, 32, dev(x), x.shape[1], x.shape[1]) for p, x in zip(_packed(lh, torch, H, [dev(w) for w in W], Ks), X)]

    def cell(sigmoid_f64):
        c, h = dev(c_prev), torch.full((B, H), float("nan"), device="cuda")
        g, d = (torch.full((B, k * H), float("nan"), device="cuda") for k in (4, 1))
        args = {}
        if addend == "column":
            args = dict(addend=dev(table), ld_addend=4 * H, addend_col=dev(col), addend_ncols=7)
        elif addend == "dense":
            args = dict(addend=dev(add), ld_addend=4 * H)
        keep = dict(gates=g, next_drop_mask=dev(drop), keep=0.8, h_drop=d) if kept else {}
        lh.load().lh_gemm_set_config_override(config)
        lh.gate_gemm_lstm_cell_packed(H, B, segs, dev(bias), c, dev(mask), c, h, sigmoid_f64=sigmoid_f64, cell_clip=clip,
                                      **args, **keep)
        torch.cuda.synchronize()
        return [t.cpu().numpy() for t in (c, h, g, d)]

    c, h, g, d = cell(f64)
    assert_close(c, c_want, "c")
    assert_close(h, h_want, "h")
    if kept:
        assert_close(g, gates_want, "gates")
        assert np.array_equal(d, (drop < np.float32(0.8)) * (np.float32(1) / np.float32(0.8)) * h)
    if f64:
        for a, b in zip((c, h) + ((g,) if kept else ()), cell(False)):
            assert np.array_equal(a[mask >= 2], b[mask >= 2])
