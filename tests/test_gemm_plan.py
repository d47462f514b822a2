"""The tile that lh_gemm takes (lh_gemm_kernel_name, no GPU needed) at sizes where one price in the cost model decides
and the choices were timed on both sides."""
import ctypes as C

import pytest

STREAMED = {(32, 32, 1, 1, 8, 64), (32, 32, 1, 1, 8, 128), (32, 64, 1, 2, 4, 64), (64, 32, 2, 1, 4, 64)}


def tile(M, N, Ks, tA=False, tX=False):
    """Tile of the kernel chosen."""
    from linmt_amd import lib
    segs = (lib.GemmSeg * len(Ks))()
    for s, K in zip(segs, Ks):
        s.A, s.lda, s.X, s.ldx, s.K = 256, K if tA else M, 256, N if tX else K, K
    name = C.create_string_buffer(128)
    lib.check(lib.load().lh_gemm_kernel_name(M, N, segs, len(Ks), tA, tX, 64 << 20, 0, name, 128), "lh_gemm_kernel_name")
    return tuple(int(v) for v in name.value.decode().split("<")[1].split(",")[:6])


@pytest.mark.parametrize("M,N,K", [(996, 109, 11516), (1692, 20, 21312), (1644, 12, 24984), (840, 130, 11896),
                                   (168, 391, 18740), (1916, 29, 29920), (2048, 64, 8192), (2048, 128, 8192)])
def test_operands_beyond_the_l2s_are_not_streamed(M, N, K):
    """Transposed A, 48 MB of operands and more: the streamed tiles took 1.1 to 1.25 times as long as a staged or
    narrow one."""
    assert tile(M, N, [K], tA=True) not in STREAMED


@pytest.mark.parametrize("M,N,K", [(1000, 64, 1000), (256, 32, 1024), (512, 48, 2048)])
def test_few_columns_of_a_small_matrix_are(M, N, K):
    """Where the operands stay in the L2s the streamed and narrow tiles are the fastest (1000 x 64, K = 1000: 8.1 us
    staged, 5.2)."""
    assert tile(M, N, [K], tA=True) in STREAMED or tile(M, N, [K], tA=True)[0] == 16


@pytest.mark.parametrize("M,N,K,tA,tX", [(246, 22, 31, False, False), (42, 64, 26, False, True), (43, 72, 31, False, True),
                                         (86, 143, 28, False, True), (1569, 112, 5590, True, False)])
def test_ragged_products_are_priced_as_staged(M, N, K, tA, tX):
    """Ragged operands take the staged form of the 32x32 tile, whose fixed part is 1.5 us more than that of the streamed
    one: 5.6 us against 5.0 at 246 x 22, K = 31; 40.9 against 36.2 at the last of these."""
    assert tile(M, N, [K], tA, tX) != (32, 32, 1, 1, 8, 128)


@pytest.mark.parametrize("M,N,K,tX", [(8830, 1538, 24, True), (22565, 673, 43, False), (21910, 298, 104, False)])
def test_large_ragged_results_of_a_short_k(M, N, K, tX):
    """64x64 tiles, 21.4, 26.8 and 22.8 us; 128x64 took 26.2, 31.1 and 25.4."""
    assert tile(M, N, [K], tX=tX) == (64, 64, 2, 2, 1, 16)


@pytest.mark.parametrize("M,N,K", [(443, 2, 120), (4567, 1, 130), (58, 47, 127)])
def test_few_ragged_columns_of_one_deep_slab(M, N, K):
    """32x32 tiles, 4.4, 5.5 and 5.9 us; 32x64, whose loads at any float's address cost it the most, 5.2, 6.4 and 6.9."""
    assert tile(M, N, [K]) == (32, 32, 1, 1, 8, 128)
