"""The projection kernel between two layers: rows' rstd as a factor of the product, rows of the result times the next weight."""
import ctypes

import pytest
import torch
from test_linear_gpu import Linear
from util import rel_err

pytestmark = pytest.mark.gpu


# tiles of every size with remainders in T, M and K; one partial sum, many, and more than are requested at once
@pytest.mark.parametrize("T,M,K,parts", [(1, 4, 8, 1), (33, 100, 72, 3), (65, 520, 1032, 33), (500, 1540, 264, 9), (700, 1000, 1096, 70),
                                         (1000, 1288, 64, 2), (1030, 3076, 136, 5), (2047, 900, 136, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_between_layers(pkg, dev, T, M, K, parts, dtype):
    L, lib = pkg._lib, pkg._lib.load()
    g = torch.Generator().manual_seed(T)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev)
    x, w, bias, res, yw = rand(T, K).to(dtype), rand(M, K).to(dtype), rand(M).to(dtype), rand(T, M), rand(M)
    ssq, eps = rand(parts, T).square() * K / parts, 1e-5
    wide = 0 if dtype == torch.float32 else 512 | 1024
    y, scaled = torch.full((T, M), float("nan"), device=dev), torch.full((T, M), float("nan"), device=dev, dtype=dtype)
    out_ssq = torch.empty((M + 31) // 32, T, device=dev)
    q = Linear(io_dtype=pkg.scan._DTYPES[dtype] | wide, T=T, M=M, K=K, x_pitch=K, y_pitch=M, x=x.data_ptr(), weight=w.data_ptr(), bias=bias.data_ptr(),
               y=y.data_ptr(), residual=res.data_ptr(), accumulate=1, y_ssq=out_ssq.data_ptr(), x_ssq=ssq.data_ptr(), ssq_parts=parts, eps=eps)
    assert lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)) == 1   # (this one wants a weight with the sums)
    L.check(lib.mpa_linear_run_scaled(ctypes.byref(q), yw.data_ptr(), scaled.data_ptr(), pkg.scan._stream(dev)), "mpa_linear_run_scaled")
    rstd = (ssq.double().sum(0) / K + eps).rsqrt()[:, None]
    want = (x.double() @ w.double().t()) * rstd + bias.double() + res.double()
    # float32 sums of at most 1096 exact products, 1 / sqrt of one ulp: 1e-5 of the largest; y * weight is rounded once more
    assert rel_err(y, want) <= 1e-5
    assert rel_err(out_ssq.sum(0), y.double().square().sum(1)) <= 1e-5
    assert torch.equal(scaled, (y * yw).to(dtype))
    # plain rows in, scaled rows out, and the other way round
    q.x_ssq = None
    L.check(lib.mpa_linear_run_scaled(ctypes.byref(q), yw.data_ptr(), scaled.data_ptr(), pkg.scan._stream(dev)), "mpa_linear_run_scaled")
    assert torch.equal(scaled, (y * yw).to(dtype))
    q.x_ssq, q.residual = ssq.data_ptr(), None
    L.check(lib.mpa_linear_run_scaled(ctypes.byref(q), None, None, pkg.scan._stream(dev)), "mpa_linear_run_scaled")
    assert rel_err(y, want - res.double()) <= 1e-5
    q.weight_kxm = 1
    assert lib.mpa_linear_run_scaled(ctypes.byref(q), None, None, pkg.scan._stream(dev)) == 2


# A residual stream whose squares are beyond float32: 1 / rms is zero, and so is the normalised row (as x * rsqrt(mean(x^2) + eps) has it),
# whatever the product of the row itself is.  An infinity makes a NaN of its row, and of that row alone.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_stack_of_huge_rows(pkg, dev, dtype):
    torch.manual_seed(0)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=3)).to(dev).to(dtype)
    with torch.no_grad():
        for layer in m.layers:
            layer.mixer.in_proj.weight.fill_(4.0)          # (a sum of the row's values is beyond float32 as well)
        x = torch.randn(1, 40, 64, device=dev).to(dtype)
        x[0, 20], x[0, 30] = 3e38, 1e25
        x[0, 35, 3] = float("inf")
        y, plain = m(x), m(x[:, :20])
    assert torch.equal(y[0, 20], x[0, 20]) and torch.equal(y[0, 30], x[0, 30])
    assert y[0, 35].isnan().all() and y[0, :35].isfinite().all()
    assert torch.equal(y[0, :20], plain[0])
