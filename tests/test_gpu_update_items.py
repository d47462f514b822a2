"""Norm and update of many tensors at once (lh_grad_sumsq_items_f32, lh_sgd_step_items_f32) against the
entry points that take one tensor, and the norms against float64: tensors of one element to more
than a launch's worth of workgroups, strided blocks, odd rows and addresses, column lists, more items
than one launch holds, a slot shared by neighbours, items without a slot, empty ones.

Tolerance of a norm: 32 squares are added in float, so 35 roundings of 2^-24 of a positive sum."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, cols, gradient rows beyond the block, offset in floats, column list
SHAPES = [(1, 1, 0, 0, False), (3, 5, 2, 0, False), (1000, 7, 3000, 0, False), (256, 64, 768, 0, True),
          (4, 2048, 12, 0, False), (8192, 1, 0, 0, False), (8196, 1, 0, 1, False), (30003, 40, 0, 0, False),
          (5, 0, 0, 0, False), (64, 33, 0, 2, True)]


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("copies", [1, 6])
def test_items_against_single_tensors(lh, shared, copies):
    rng = np.random.default_rng(copies + 10 * shared)
    L = lh.load()
    shapes = SHAPES * copies
    items, keep = (lh.UpdateItem * len(shapes))(), []
    scale, lr, clip = 0.25, 0.1, 3.0
    for i, (rows, cols, extra, off, listed) in enumerate(shapes):
        ldg, ldt = rows + extra, rows + extra
        g = torch.from_numpy(rng.normal(0, 1, off + ldg * max(cols, 1)).astype(np.float32)).cuda()
        n_t = 2 * cols if listed else max(cols, 1)
        t = torch.from_numpy(rng.normal(0, 1, off + ldt * n_t).astype(np.float32)).cuda()
        idx = torch.from_numpy(rng.permutation(n_t)[:cols].astype(np.int32)).cuda() if listed else None
        norm = 0 if shared else (-1 if i % 7 == 3 else i)
        keep.append((g, t, idx, rows, cols, ldg, ldt, off, norm))
        items[i] = lh.UpdateItem(t[off:].data_ptr(), ldt, g[off:].data_ptr(), ldg, rows, cols,
                                 idx.data_ptr() if listed else None, norm)
    singles = [(g.clone(), t.clone()) for g, t, *_ in keep]
    stream = torch.cuda.current_stream().cuda_stream
    ws = torch.full((L.lh_grad_sumsq_items_workspace(items, len(shapes)),), float("nan"), dtype=torch.float64, device="cuda")
    norms = torch.zeros(len(shapes), dtype=torch.float64, device="cuda")
    lh.check(L.lh_grad_sumsq_items_f32(items, len(shapes), scale, ws.data_ptr(), norms.data_ptr(), stream), "norms")
    want = np.zeros(len(shapes))
    for g, _, _, rows, cols, ldg, _, off, norm in keep:
        if norm >= 0 and cols:
            block = g.cpu().numpy()[off: off + ldg * cols].reshape(cols, ldg)[:, :rows].astype(np.float64)
            want[norm] += (scale * block * block * scale).sum()
    assert np.all(np.abs(norms.cpu().numpy() - want) <= 35 * 2.0 ** -24 * want)
    lh.check(L.lh_sgd_step_items_f32(items, len(shapes), lr, scale, norms.data_ptr(), clip, 0.5, stream), "update")
    for (g, t, idx, rows, cols, ldg, ldt, off, norm), (g1, t1) in zip(keep, singles):
        lh.check(L.lh_sgd_step_f32(t1[off:].data_ptr(), ldt, g1[off:].data_ptr(), ldg, rows, cols,
                                   None if idx is None else idx.data_ptr(), lr, scale,
                                   norms[norm:].data_ptr() if norm >= 0 else None, clip, 0.5, stream), "single")
        assert torch.equal(t, t1) and torch.equal(g, g1), (rows, cols)   # gradients cleared, gaps untouched


def test_items_refused(lh):
    L = lh.load()
    x = torch.zeros(64, device="cuda")
    d = torch.zeros(8, dtype=torch.float64, device="cuda")

    def item(norm, ld=4):
        return lh.UpdateItem(x.data_ptr(), ld, x.data_ptr(), ld, 4, 2, None, norm)

    apart = (lh.UpdateItem * 3)(item(0), item(1), item(0))
    assert L.lh_grad_sumsq_items_f32(apart, 3, 1.0, d.data_ptr(), d.data_ptr(), C.c_void_p(0)) != 0
    short = (lh.UpdateItem * 1)(item(0, ld=3))
    assert L.lh_grad_sumsq_items_f32(short, 1, 1.0, d.data_ptr(), d.data_ptr(), C.c_void_p(0)) != 0
    assert L.lh_sgd_step_items_f32(short, 1, 1.0, 1.0, d.data_ptr(), 1.0, 0.0, C.c_void_p(0)) != 0
    fine = (lh.UpdateItem * 1)(item(0))
    assert L.lh_sgd_step_items_f32(fine, 1, 1.0, 1.0, None, 1.0, 0.0, C.c_void_p(0)) != 0
