"""Which of the pipelined GEMM tiles the planner takes for large products.  No GPU."""
import ctypes

import pytest

from chestnut import _lib


@pytest.mark.parametrize('kn', [0, 1])
@pytest.mark.parametrize('M,N,K,tile', [
    (4096, 4096, 4096, 9),     # two waves of 256x128, four of 128x128
    (2048, 4096, 2048, 9),     # one wave of 256x128, two of 128x128
    (1536, 4096, 2048, 9),     # 192 of 256x128, 384 of 128x128
    (2048, 2048, 2048, 1),     # one wave of 128x128
    (1000, 2184, 1984, 1)])
def test_planner_takes_the_tile_with_the_cheapest_waves(kn, M, N, K, tile):
    t, s, nb = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_size_t()
    _lib.call('ck_gemm_workspace', M, N, K, kn, ctypes.byref(t), ctypes.byref(s), ctypes.byref(nb))
    assert (t.value, s.value, nb.value) == (tile, 1, 0)


def test_planner_keeps_an_asked_split():
    t, s, nb = ctypes.c_int(0), ctypes.c_int(2), ctypes.c_size_t()
    _lib.call('ck_gemm_workspace', 4096, 4096, 4096, 0, ctypes.byref(t), ctypes.byref(s), ctypes.byref(nb))
    assert (t.value, s.value, nb.value) == (1, 2, 2 * 4096 * 4096 * 4)
