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


def _packed_plan(lib, H, B, Ks):
    segs = (lib.GemmSeg * 3)()
    for s, K in zip(segs, Ks):
        s.A, s.lda, s.X, s.ldx, s.K = 256, 4 * H, 256, K, K
    faster, name = C.c_int(), C.create_string_buffer(128)
    lib.check(lib.load().lh_gate_gemm_lstm_cell_packed_plan(H, B, segs, len(Ks), 1, 64 << 20, C.byref(faster), name, 128),
              "lh_gate_gemm_lstm_cell_packed_plan")
    return name.value.decode() if faster.value else None


@pytest.mark.parametrize("H,B,Ks,packed", [(1084, 134, (1084, 1084), True), (1000, 64, (1000, 1000), True),
                                           (2048, 128, (2048, 2048), False), (2048, 192, (2048, 2048), False)])
def test_packed_matrices_by_time_not_by_workgroups(H, B, Ks, packed):
    """More workgroups than CUs are no reason by themselves: the first of these is 544 and took 43.8 us packed, 46.5 from
    the stored matrix; the last two took 92.8 and 82.6, 126.6 and 122.6."""
    from linmt_amd import lib
    assert (_packed_plan(lib, H, B, Ks) is not None) == packed


@pytest.mark.parametrize("H,B,Ks", [(1956, 58, (1956, 1956)), (1364, 60, (1364, 1364, 1364)), (1740, 44, (1740, 1740, 1740))])
def test_large_stored_matrices_are_not_streamed(H, B, Ks):
    """A tile's share of a stored gate matrix is 32-byte runs: streamed from HBM it took 1.36 times the time of the L2s (the
    first of these 69 us, 51 as a split product with the cell kernel behind it)."""
    from linmt_amd import lib
    assert _plan(lib, H, B, Ks) != "gate_gemm_cell_kernel<64, 32, 2, 1, 4, 64>"
