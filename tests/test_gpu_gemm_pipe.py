"""The pipelined GEMM tiles (1: 128x128, 9: 256x128, 16:
64x64) and the 32x32 tile with K over the waves (17) against the
oracle where they can go wrong: one K-step up to more than the ring holds,
ragged M and N around a tile edge, M-tile counts that do not fill a group of
four, split K, outputs the 16-byte stores do not fit, every epilogue, B as
[N][K] and [K][N].  Bounds: the f32 summation error of tests/test_gpu_kernels.py."""
import ctypes

import numpy as np
import pytest

from oracle import kernels as OK
from test_gpu_kernels import _gemm_check, dev, host

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def tiles_for(shapes, kn_of, split_of):
    """(tile, *shape) of every tile and shape that go together: tile 17 takes B as
    [N][K] and no split."""
    return [(t, *s) for s in shapes for t in (1, 9, 16, 17) if t != 17 or not kn_of(s) and split_of(s) == 1]


TAILS = [
    (1, 8, 64, 1),            # one row, one 16-byte column chunk, one K-step
    (257, 264, 128, 1),       # one past the 256 edge
    (255, 120, 192, 1),       # one short of it
    (129, 136, 256, 1), (300, 520, 320, 1), (130, 128, 448, 1),   # around the 3- and 4-stage rings
    (1290, 392, 128, 1),      # 11 and 6 M-tiles: last group of four not full
    (33, 40, 704, 1), (31, 24, 768, 1), (65, 72, 832, 1), (63, 56, 896, 1),   # 11 to 14 steps: each tail of the steps in fours
    (65, 72, 640, 1), (63, 56, 576, 1),   # around a 64 edge; 10 and 9 steps (odd and even tails of the step pairs)
    (300, 520, 1024, 4), (128, 256, 384, 3)]


@pytest.mark.parametrize('tile,kn,M,N,Kd,split', tiles_for([(kn, *s) for kn in (False, True) for s in TAILS],
                                                           lambda s: s[0], lambda s: s[4]))
def test_pipe_tiles_tails(gpu, tile, kn, M, N, Kd, split):
    from chestnut import kernels as K
    print(f'[gemm] pipe tile {tile} kn={kn} {M}x{N}x{Kd} split {split}', flush=True)
    rng = np.random.default_rng(M + N + Kd + tile)
    A = rng.standard_normal((M, Kd)).astype(np.float16)
    B = rng.standard_normal((Kd, N) if kn else (N, Kd)).astype(np.float16)
    b = rng.standard_normal(N).astype(np.float32)
    C = host(K.gemm(dev(gpu, A), dev(gpu, B), b_kn=kn, bias=dev(gpu, b), tile=tile, split_k=split))
    _gemm_check(C - b, A, B, transB=not kn, depth=Kd // 16 + 40)


@pytest.mark.parametrize('tile,kn,N,ldc,split', tiles_for(
    [(kn, N, ldc, split) for kn, N, ldc in [(False, 201, 201), (False, 200, 203), (True, 200, 203)] for split in (1, 2)],
    lambda s: s[0], lambda s: s[3]))
def test_pipe_tiles_without_16_byte_stores(gpu, tile, kn, N, ldc, split):
    """N odd, or a row pitch that is no multiple of 16 bytes: stored per
    element, and nothing outside [M][N] written."""
    from chestnut import _lib
    torch = gpu
    M, Kd = 150, 256
    rng = np.random.default_rng(N + ldc)
    A = rng.standard_normal((M, Kd)).astype(np.float16)
    B = rng.standard_normal((Kd, N) if kn else (N, Kd)).astype(np.float16)
    Ad, Bd = dev(torch, A), dev(torch, B)
    C = torch.full((M, ldc), 7.0, device='cuda')
    ws = torch.empty(split * M * N, device='cuda')
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.call('ck_gemm', p(Ad), p(Bd), p(C), None, M, N, Kd, Kd, N if kn else Kd, ldc, 1 if kn else 0, tile, split,
              p(ws), ws.numel() * 4, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    got = host(C)
    _gemm_check(got[:, :N], A, B, transB=not kn)
    assert (got[:, N:] == 7.0).all()


@pytest.mark.parametrize('tile,M,N,split', tiles_for([(200, 264, 1), (200, 260, 1), (130, 264, 2)],
                                                     lambda s: False, lambda s: s[2]))
@pytest.mark.parametrize('epi', [1, 2, 3, 4])
def test_pipe_tiles_epilogues(gpu, tile, M, N, split, epi):
    from chestnut import kernels as K
    torch = gpu
    rng = np.random.default_rng(epi + N)
    Kd = 256
    A = (rng.standard_normal((M, Kd)) / 8).astype(np.float16)
    W = (rng.standard_normal((N, Kd)) / 8).astype(np.float16)
    b = rng.standard_normal(N).astype(np.float32)
    acc = OK.gemm(A, W, transB=True) + b
    if epi == 4:
        C0 = rng.standard_normal((M, N)).astype(np.float32)
        out = dev(torch, C0.copy())
        K.gemm_epi(dev(torch, A), dev(torch, W), dev(torch, b), 4, out, tile=tile, split_k=split)
        scale = np.abs(A.astype(np.float64)) @ np.abs(W.astype(np.float64)).T + np.abs(b) + np.abs(C0)
        assert np.all(np.abs(host(out) - (C0 + acc)) <= (Kd // 16 + 40) * U * scale)
        return
    out = torch.empty(M, N, dtype=torch.float16, device='cuda')
    K.gemm_epi(dev(torch, A), dev(torch, W), dev(torch, b), epi, out, tile=tile, split_k=split)
    ref = {1: lambda v: v, 2: lambda v: np.maximum(v, 0), 3: OK.gelu}[epi](acc)
    ref = ref.astype(np.float32).astype(np.float16).astype(np.float64)
    # one f16 rounding of an f32 value within reassociation noise: at most one ulp apart
    ulp = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float64)
    assert np.all(np.abs(host(out).astype(np.float64) - ref) <= ulp + 1e-7)


@pytest.mark.parametrize('tile', [1, 9, 16])
@pytest.mark.parametrize('epi,M,N', [(4, 16400, 32776), (1, 32792, 32776)])
def test_pipe_tiles_output_of_2_gib(gpu, tile, epi, M, N):
    """Outputs whose offsets do not fit the 32-bit buffer stores leave by
    non-temporal ones: the first and last rows, the rows around 2 GiB and some
    between, against 64-bit sums."""
    from chestnut import kernels as K
    torch = gpu
    Kd, el = 64, 4 if epi == 4 else 2
    assert el * M * N > 1 << 31
    g = torch.Generator(device='cuda')
    g.manual_seed(M + tile)
    A = (torch.randn(M, Kd, generator=g, device='cuda') / 8).half()
    W = (torch.randn(N, Kd, generator=g, device='cuda') / 8).half()
    b = torch.randn(N, generator=g, device='cuda')
    at = (1 << 31) // (el * N)
    rows = torch.tensor(sorted({0, 1, 255, 256, M // 3, at - 1, at, at + 1, M - 2, M - 1}), device='cuda')
    print(f'[gemm] 2 GiB output, tile {tile} epi {epi} {M}x{N}', flush=True)
    out = torch.zeros(M, N, dtype=torch.float32 if epi == 4 else torch.float16, device='cuda')
    if epi == 4:
        out[rows] = 3.0
    K.gemm_epi(A, W, b, epi, out, tile=tile, split_k=1)
    Wt = W.double().t().contiguous()
    ref = A[rows].double() @ Wt + b.double() + (3.0 if epi == 4 else 0.0)
    scale = A[rows].double().abs() @ Wt.abs() + b.double().abs() + 3.0
    err = (Kd // 16 + 40) * U * scale + (0 if epi == 4 else 2.0 ** -11 * ref.abs() + 2.0 ** -25)
    assert bool(((out[rows].double() - ref).abs() <= err).all())
    # and every other row was written: none is left as it was
    assert bool((out.count_nonzero(dim=1) > N // 2).all())
