"""Which kernel the rules give launches to, without a GPU (the rules then take 256 compute units)."""
import ctypes

import pytest

from megablocks_amd import _lib

FEW, GENERAL, FEW_TILES = 0, 1, 2
PLAIN, ACT, DACT, DGATE, GATE, COMBINE = 0, 1, 2, 3, 5, 7


@pytest.fixture
def kernel():
    f = _lib.lib.mbx_debug_row_kernel_by_rule
    f.argtypes = [ctypes.c_int] * 4 + [ctypes.c_int64] + [ctypes.c_int] * 3

    def ask(layout, experts, rows, k, n, epi=PLAIN, dual=False, workspace=True):
        return f(layout, epi, dual, experts, experts * rows, k, n, workspace)
    return ask


@pytest.mark.parametrize('layout,experts,rows,k,n,epi', [
    (_lib.NT, 4, 500, 1408, 2048, PLAIN), (_lib.NT, 8, 3234, 576, 72, PLAIN), (_lib.NT, 160, 52, 704, 320, PLAIN),
    (_lib.NN, 8, 500, 1408, 512, PLAIN), (_lib.NT, 32, 43, 3176, 152, GATE), (_lib.NT, 16, 1530, 1536, 88, DACT),
    # more than 64 experts
    (_lib.NT, 95, 132, 640, 3136, DACT), (_lib.NT, 87, 125, 640, 3328, DACT), (_lib.NT, 194, 80, 1208, 1600, DACT), (_lib.NT, 103, 61, 2688, 704, ACT),
    (_lib.NT, 126, 52, 400, 6080, DGATE), (_lib.NT, 128, 92, 576, 4352, DGATE), (_lib.NT, 78, 102, 384, 1728, PLAIN),
    # more than eight rounds: few rows, the activation's gradient, narrow products
    (_lib.NT, 151, 67, 320, 5504, ACT), (_lib.NT, 105, 137, 576, 8000, ACT), (_lib.NT, 97, 10059, 128, 64, PLAIN),
    # a long reduction next to a mostly empty wide tile
    (_lib.NN, 36, 825, 7768, 64, PLAIN),
    # half-height tiles whose last round two short parts would not shorten
    (_lib.NN, 64, 227, 1216, 1344, PLAIN)])
def test_launches_of_few_tiles(kernel, layout, experts, rows, k, n, epi):
    """Measured 6 - 50 % shorter in the kernel for few tiles than in the general one."""
    assert kernel(layout, experts, rows, k, n, epi) == FEW_TILES


@pytest.mark.parametrize('layout,experts,rows,k,n,epi,dual', [
    (_lib.NT, 8, 13673, 128, 4328, GATE, False), (_lib.NT, 2, 15001, 128, 8848, GATE, False), (_lib.NT, 16, 17159, 128, 2960, ACT, False),
    (_lib.NT, 128, 759, 256, 2824, ACT, False), (_lib.NT, 64, 353, 64, 13432, PLAIN, False), (_lib.NT, 90000, 1, 64, 4096, PLAIN, False),
    (_lib.NN, 8, 2037, 9536, 240, PLAIN, False), (_lib.NN, 4, 1705, 10880, 752, PLAIN, False), (_lib.NN, 32, 288, 12512, 400, PLAIN, True),
    (_lib.NT, 2903, 62, 176, 160, PLAIN, False), (_lib.NT, 2275, 169, 192, 136, DACT, False), (_lib.NN, 147, 271, 6848, 160, PLAIN, False)])
def test_launches_outside_of_what_the_estimates_hold_for(kernel, layout, experts, rows, k, n, epi, dual):
    """Measured 5 - 45 % longer in the kernel for few tiles than in the general one, or of the same kind."""
    assert kernel(layout, experts, rows, k, n, epi, dual) in (FEW, GENERAL)


@pytest.mark.parametrize('experts,rows,k,n', [(4, 104, 13120, 512), (4, 151, 14016, 1600), (12, 61, 8640, 512), (8, 217, 7872, 576), (4, 1200, 8640, 120)])
def test_combines_whose_tails_are_cut_are_judged_so(kernel, experts, rows, k, n):
    """Measured 10 - 55 % shorter in the general kernel, which cuts them along the reduction as it does the plain product; without a workspace
    nothing is cut, and the kernel for few tiles takes them."""
    assert kernel(_lib.NN, experts, rows, k, n, COMBINE) == kernel(_lib.NN, experts, rows, k, n, PLAIN) == GENERAL
    assert kernel(_lib.NN, experts, rows, k, n, COMBINE, workspace=False) == FEW_TILES


ROUNDS_OF_256, TILES_128, TILES_256_128, TILES_128_AHEAD = 0, 1, 2, 3


@pytest.mark.parametrize('experts,rows,k,n,want', [
    # whole 64-byte pieces, or few columns: fetched ahead, 256 x 128 tiles for many
    (64, 64, 1024, 4096, TILES_128_AHEAD), (59, 35, 2376, 1728, TILES_128_AHEAD), (64, 128, 1024, 4096, TILES_256_128), (27, 72, 696, 7904, TILES_256_128),
    (64, 1, 1024, 4096, TILES_128_AHEAD), (55, 121, 2568, 208, TILES_128_AHEAD), (54, 122, 4320, 1016, TILES_256_128), (4, 1, 8, 8, TILES_128_AHEAD),
    # pieces that two of many tiles store parts of: neither, up to 128 rows
    (59, 35, 2376, 1736, TILES_128), (9, 63, 5576, 5736, TILES_128), (27, 72, 696, 7912, TILES_128), (52, 82, 1400, 1832, TILES_128),
    (69, 128, 872, 5112, TILES_128), (69, 129, 920, 5112, TILES_256_128), (69, 200, 360, 5112, TILES_128_AHEAD),
    # above 512 rows no 128 x 128 tiles out of estimates
    (54, 755, 176, 6184, TILES_256_128), (93, 648, 1392, 216, TILES_256_128), (64, 300, 1408, 512, TILES_128_AHEAD), (8, 1024, 576, 1024, TILES_128_AHEAD),
    (64, 2000, 1024, 4096, ROUNDS_OF_256)])
def test_weight_gradients_of_few_rows(experts, rows, k, n, want):
    """On the far side of the lines between them the kernels were measured 5 - 30 % longer."""
    f = _lib.lib.mbx_debug_tn_kernel_by_rule
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    assert f(experts, experts * rows, k, n) == want


@pytest.mark.parametrize('experts,rows,k,n,small', [
    (64, 64, 1408, 1024, True), (64, 100, 1408, 1024, False), (8, 256, 1408, 512, True), (1, 0, 64, 64, True), (8, 1024, 1024, 4096, False),
    # the small tile for less padding, in short reductions from a quarter on, in long ones from 45 %
    (28, 726, 320, 320, True), (68, 101, 288, 816, True), (19, 768, 2496, 320, False), (45, 165, 8192, 320, True), (106, 103, 192, 1024, False)])
def test_fp32_tiles(experts, rows, k, n, small):
    f = _lib.lib.mbx_debug_f32_small_by_rule
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    assert bool(f(experts, experts * rows, k, n, 0)) == small
