"""The tile that lh_gate_gemm_lstm_cell_f32 takes (lh_gate_gemm_lstm_cell_plan, no GPU needed): a few columns of a
small or medium hidden size leave most CUs empty, and of all shapes the 32 x 32 tile with eight wavefronts along K is
within 10 % of the fastest there (sweep over 64 to 640 hidden units, 1 to 64 columns, 1 to 3 segments).  The choice
must not depend on which side of some size the model lies."""
import ctypes as C

import pytest


def _plan(lib, H, B, Ks):
    segs = (lib.GemmSeg * 3)()
    for s, K in zip(segs, Ks):
        s.A, s.lda, s.X, s.ldx, s.K = 256, 4 * H, 256, K, K
    fusable, name = C.c_int(), C.create_string_buffer(128)
    lib.check(lib.load().lh_gate_gemm_lstm_cell_plan(H, B, segs, len(Ks), 0, 64 << 20, C.byref(fusable), name, 128),
              "lh_gate_gemm_lstm_cell_plan")
    return name.value.decode() if fusable.value else None


@pytest.mark.parametrize("segments,widest", [(1, 640), (2, 512), (3, 320)])
@pytest.mark.parametrize("B", [1, 5, 12, 32, 64])
def test_few_columns_take_one_shape(segments, widest, B):
    from linmt_amd import lib
    names = {_plan(lib, H, B, (H,) * segments) for H in range(64, widest + 1, 4)}
    assert names <= {"gate_gemm_cell_kernel<32, 32, 1, 1, 8, 64>", "gate_gemm_cell_kernel<32, 32, 1, 1, 8, 128>"}, names
