"""Per-tile time stamps of the grouped products (`bench.py --tile-ticks`)."""
import ctypes
import os

import pytest
import torch

import bench

TICKS_LIBRARY = os.path.join(os.path.dirname(os.path.abspath(bench.__file__)), 'megablocks_amd', 'libmbx_ticks.so')


def test_tile_phases():
    t = torch.zeros(4, 3, 8, dtype=torch.float64)
    assert bench.tile_phases(t) == {'tiles': 0, 'note': 'no stamped tiles'}
    for tile, start in ((0, 100.0), (1, 112.0)):   # one workgroup, two tiles
        t[2, tile] = start + torch.tensor([0.0, 3.0, 8.0, 2.0, 9.0, 10.0, 0.5, 1.0], dtype=torch.float64)
    got = bench.tile_phases(t)
    assert got['tiles'] == 2 and got['workgroups'] == 1 and got['start_to_first_k_tile'] == 3.0 and got['main_loop'] == 5.0
    assert got['between_tiles_of_a_workgroup'] == 2.0 and got['tile_total'] == 10.0
    assert got['first_tile_start_to_last_tile_end_ms'] == 0.022


@pytest.mark.gpu
@pytest.mark.parametrize('groups,rows,k,n', [(64, 256, 256, 128), (64, 2, 128, 1024), (64, 24, 128, 2048)])
def test_every_16_bit_launch_is_stamped(groups, rows, k, n):
    """Also the launches that the product library gives to kernels without stamps, for a few rows per expert."""
    from megablocks_amd import _lib
    lib = ctypes.CDLL(TICKS_LIBRARY)
    lib.mbx_debug_set_ticks.argtypes = [ctypes.c_void_p]
    lib.mbx_gmm.argtypes = _lib.lib.mbx_gmm.argtypes
    total = groups * rows
    a = torch.randn(total, k, device='cuda').bfloat16()
    d = torch.randn(total, n, device='cuda').bfloat16()
    w = torch.randn(groups, n, k, device='cuda').bfloat16()
    bins = torch.arange(1, groups + 1, device='cuda', dtype=torch.int32) * rows
    ticks = torch.zeros(16384 * 64 * 8, dtype=torch.int64, device='cuda')   # kTickWorkgroups, kTickTiles, kTickIds of gmm_dma.h
    for layout, x, y, out in ((_lib.NT, a, w, torch.empty_like(d)), (_lib.NN, d, w, torch.empty_like(a)),
                              (_lib.TN, a, d, torch.empty(groups, k, n, device='cuda', dtype=torch.bfloat16))):
        inner, outer = (n, k) if layout == _lib.NN else (k, n)
        ticks.zero_()
        torch.cuda.synchronize()
        assert lib.mbx_debug_set_ticks(ticks.data_ptr()) == 0
        assert lib.mbx_gmm(x.data_ptr(), y.data_ptr(), out.data_ptr(), _lib.dtype_of(x), bins.data_ptr(), groups, total, inner, outer,
                           layout, _lib.stream()) == 0
        torch.cuda.synchronize()
        assert lib.mbx_debug_set_ticks(None) == 0
        assert bench.tile_phases(ticks.view(16384, 64, 8).cpu().double() / 100.0)['tiles'] >= groups
