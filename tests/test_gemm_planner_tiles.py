"""Which GEMM tile the planner takes where 128x128 tiles number 64 or more, which
for a [K][N] B of a small product, and the swizzle of a 64-column [K][N] stage
(CPU replay of gemm_pipe.hip).  No GPU."""
import ctypes

import numpy as np
import pytest

from chestnut import _lib
from test_bt_layout import tr_read


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


@pytest.mark.parametrize('M,N,K,kn,tile,split', [
    (1000, 1000, 1024, 0, 16, 1),     # 64 tiles of 128x128 would split K and reduce
    (1000, 1000, 128, 0, 4, 1),       # two K-steps
    (1000, 1000, 128, 1, 16, 1),
    (221, 4120, 64, 0, 4, 1),         # 66 of 128x128, 260 of 64x64
    (1504, 1504, 1536, 0, 1, 1),      # 144 of 128x128 for 24 K-steps
    (200, 520, 2048, 0, 17, 1),       # few tiles, long K: 32x32 instead of a split in 4
    (11, 6272, 832, 0, 17, 1), (16, 4096, 4096, 0, 17, 1), (64, 8192, 512, 0, 4, 1),
    (256, 2048, 512, 0, 4, 1),        # 512 tiles of 32x32
    (64, 512, 4096, 0, 4, 16), (40, 40, 8192, 0, 4, 16),   # splits with more chains of roundings
    (11, 6272, 832, 1, 16, 1),        # few rows: B read as it lies
    (16, 4096, 4096, 1, 16, 4),
    (40, 40, 8192, 1, 16, 16),
    (9000, 40, 256, 1, 16, 1), (40, 9000, 256, 1, 16, 1)])
def test_planner_small_tiles(M, N, K, kn, tile, split):
    t, s, nb = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_size_t()
    _lib.call('ck_gemm_workspace', M, N, K, kn, ctypes.byref(t), ctypes.byref(s), ctypes.byref(nb))
    assert (t.value, s.value, nb.value) == (tile, split, 4 * split * M * N if split > 1 else 0)


def test_planner_keeps_an_asked_split():
    t, s, nb = ctypes.c_int(0), ctypes.c_int(2), ctypes.c_size_t()
    _lib.call('ck_gemm_workspace', 4096, 4096, 4096, 0, ctypes.byref(t), ctypes.byref(s), ctypes.byref(nb))
    assert (t.value, s.value, nb.value) == (1, 2, 2 * 4096 * 4096 * 4)


def test_64_column_stage_gives_the_mfma_b_operand():
    """4 waves fill a [64][64] stage with 1 KB loads (8 rows each); wave column
    wn reads its 32 columns as one fragment per 16-row slice: lane l gets column
    l % 32, k 8 (l / 32) .. +7, no bank twice in a 16-lane pass."""
    BN, BK, NW = 64, 64, 4

    def swz(r):
        return ((r >> 1) & 3) << 1

    B = np.arange(BK * BN).reshape(BK, BN)
    lds = np.full(BK * BN, -1, np.int64)
    nib = BN // (8 * NW)
    for wave in range(NW):
        for i in range(nib):
            for lane in range(64):
                c = (wave * nib + i) * 64 + lane
                r, q = c // 8, (c % 8) ^ swz(c // 8)
                lds[c * 8:c * 8 + 8] = B[r, q * 8:q * 8 + 8]
    assert (lds >= 0).all()
    for wn in range(2):
        for kk in range(4):
            half = []
            for h in range(2):
                offs = []
                for lane in range(64):
                    g, a, b = lane >> 4, (lane >> 2) & 3, lane & 3
                    row, col = 8 * (g >> 1) + 4 * h + a, wn * 32 + 16 * (g & 1) + 4 * b
                    offs.append(row * BN + (((col >> 3) ^ swz(row)) << 3) + (col & 7) + kk * 16 * BN)
                half.append(tr_read(lds, offs))
                for g in range(4):
                    banks = np.concatenate([(2 * np.array(offs[16 * g:16 * g + 16]) // 4) % 64 + d for d in (0, 1)])
                    assert np.bincount(banks, minlength=64).max() <= 1
            frag = np.concatenate(half, axis=1)
            for lane in range(64):
                k0, n = kk * 16 + 8 * (lane // 32), wn * 32 + lane % 32
                assert (frag[lane] == B[k0:k0 + 8, n]).all()
