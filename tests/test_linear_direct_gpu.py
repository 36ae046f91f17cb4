"""The projection kernel (csrc/linear.hip) with rows that go to LDS directly: numbers of stages around those in flight, ends of K within a
stage and within a row's padding, ends of T and M within a tile, and the sizes at which its tiles change."""
import ctypes

import pytest
import torch

from test_linear_gpu import Linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,M,K,pad", [
    (1, 4, 8, 0), (1, 36, 64, 8), (65, 132, 72, 0), (63, 100, 128, 16), (64, 128, 136, 0), (70, 132, 192, 8), (33, 64, 200, 0), (64, 32, 256, 8),
    (40, 64, 320, 0), (129, 260, 448, 8), (31, 36, 520, 0), (200, 68, 776, 8),    # one to seven stages of a share, one to four shares of K
    (300, 2560, 264, 0), (1400, 772, 1032, 8), (1400, 420, 1032, 0),               # 64 x 128; more than one round of 64 x 64 and of 64 x 32
    (400, 640, 1280, 0), (700, 392, 784, 8), (3000, 80, 264, 0),                   # 64 x 32, where 32 x 32 are more than a round
    (1100, 1540, 136, 0), (8200, 516, 72, 0),                                      # 128 x 128; W walked first
])
def test_products_against_float64(pkg, dev, dtype, T, M, K, pad):
    L = pkg._lib
    lib = L.load()
    torch.manual_seed(T + M + K)
    x = torch.full((T + 1, K + pad), float("nan"), dtype=dtype, device=dev)     # rows and columns that are not to be read
    x[:T, :K] = torch.randn(T, K, device=dev).to(dtype)
    w = torch.full((M + 1, K), float("nan"), dtype=dtype, device=dev)
    w[:M] = torch.randn(M, K, device=dev).to(dtype)
    y = torch.zeros(T, M, dtype=dtype, device=dev)
    q = Linear(io_dtype=pkg.scan._DTYPES[dtype], T=T, M=M, K=K, x_pitch=K + pad, y_pitch=M, x=x.data_ptr(), weight=w.data_ptr(), y=y.data_ptr())
    L.check(lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)), "mpa_linear_run")
    xd, wd = x[:T, :K].double().cpu(), w[:M].double().cpu()
    ref = xd @ wd.t()
    # float32 sums: K roundings of 2^-24 of the sum of magnitudes; a bfloat16 result is rounded once
    bound = (K + 2) * 2.0 ** -24 * (xd.abs() @ wd.abs().t()) + (2.0 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0)
    assert ((y.double().cpu() - ref).abs() <= bound).all()
    # and with the rows' factor: sums of squares that are one
    ssq = torch.full((2, T), K / 2, device=dev)
    q.x_ssq, q.ssq_parts, q.eps = ssq.data_ptr(), 2, 0.0
    y2 = torch.zeros_like(y)
    q.y = y2.data_ptr()
    L.check(lib.mpa_linear_run_scaled(ctypes.byref(q), None, None, pkg.scan._stream(dev)), "mpa_linear_run_scaled")
    assert ((y2.double().cpu() - ref).abs() <= 2 * bound + 2.0 ** -20 * ref.abs()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,M,K,pitch", [(2, 4, 264, 1 << 27), (3, 36, 64, 89478480), (2, 4, (1 << 24) - 8, (1 << 24) - 8)])
def test_pitches_of_which_a_tile_has_more_than_32_bits(pkg, dev, dtype, T, M, K, pitch):
    """Sums of whole numbers up to 2^24, exact in any order."""
    L = pkg._lib
    lib = L.load()
    torch.manual_seed(M)
    x = torch.empty((T - 1) * pitch + K, dtype=dtype, device=dev).as_strided((T, K), (pitch, 1))
    x.copy_(torch.randint(-1, 2, (T, K), device=dev))
    w = torch.randint(-1, 2, (M, K), device=dev).to(dtype)
    y = torch.zeros(T, M, dtype=dtype, device=dev)
    q = Linear(io_dtype=pkg.scan._DTYPES[dtype], T=T, M=M, K=K, x_pitch=pitch, y_pitch=M, x=x.data_ptr(), weight=w.data_ptr(), y=y.data_ptr())
    L.check(lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)), "mpa_linear_run")
    want = torch.stack([torch.stack([(a.float() * b.float()).sum(dtype=torch.float64) for b in w]) for a in x])
    assert torch.equal(y, want.to(dtype))
