"""The projection kernel of short sequences against float64 products."""
import ctypes

import pytest
import torch
from util import TOL, rel_err

pytestmark = pytest.mark.gpu


class Linear(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int64) for n in ("T", "M", "K", "x_pitch", "y_pitch")] + \
               [(n, ctypes.c_void_p) for n in ("x", "weight", "bias", "y", "norm_weight", "x_ssq")] + \
               [("ssq_parts", ctypes.c_int64), ("eps", ctypes.c_float), ("io_dtype", ctypes.c_int32), ("weight_kxm", ctypes.c_int32), ("accumulate", ctypes.c_int32), ("residual", ctypes.c_void_p), ("y_ssq", ctypes.c_void_p)]


# tiles of every size (few to many rows and columns, short and long K) with remainders in T, M and K
@pytest.mark.parametrize("T,M,K,pitch", [(1, 4, 8, 8), (33, 100, 72, 80), (65, 520, 1032, 1032), (500, 1540, 264, 264), (700, 1000, 1096, 1096),
                                         (1000, 1288, 64, 128), (2047, 900, 136, 144)])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_matches_product(pkg, dev, T, M, K, pitch, fused, dtype):
    L, lib = pkg._lib, pkg._lib.load()
    g = torch.Generator().manual_seed(T)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev)
    x, w = rand(T, pitch).to(dtype), rand(M, K).to(dtype)
    q = Linear(io_dtype=pkg.scan._DTYPES[dtype], T=T, M=M, K=K, x_pitch=pitch, y_pitch=M, x=x.data_ptr(), weight=w.data_ptr())
    y = torch.full((T, M), float("nan"), device=dev, dtype=dtype)
    q.y = y.data_ptr()
    want = x[:, :K].double() @ w.double().t()
    if fused:
        bias, res, nw = rand(M).to(dtype), rand(T, M).to(dtype), rand(K)
        ssq, eps = rand(5, T).square() * K / 5, 1e-5
        out_ssq = torch.empty((M + 31) // 32, T, device=dev)
        q.bias, q.residual, q.y_ssq = bias.data_ptr(), res.data_ptr(), out_ssq.data_ptr()
        q.norm_weight, q.x_ssq, q.ssq_parts, q.eps = nw.data_ptr(), ssq.data_ptr(), 5, eps
        normed = x[:, :K].double() * (ssq.double().sum(0) / K + eps).rsqrt()[:, None] * nw.double()
        want = normed @ w.double().t() + bias.double() + res.double()
    L.check(lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)), "mpa_linear_run")
    assert rel_err(y.float(), want) <= TOL[dtype]  # (bfloat16: rounded twice with a residual)
    if fused:
        assert rel_err(out_ssq.sum(0), y.double().square().sum(1)) <= 1e-5


@pytest.mark.parametrize("T,M,K,pitch", [(1, 8, 8, 8), (33, 104, 72, 80), (65, 520, 1032, 1032), (500, 1544, 264, 264), (700, 1000, 1096, 1096),
                                         (1000, 1288, 64, 128), (2047, 904, 136, 144)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_with_the_weight_transposed(pkg, dev, T, M, K, pitch, dtype):
    L, lib = pkg._lib, pkg._lib.load()
    g = torch.Generator().manual_seed(M)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev).to(dtype)
    x, w, y = rand(T, pitch), rand(K, M), rand(T, M + 8)
    want = x[:, :K].double() @ w.double() + y[:, :M].double()
    pad = y[:, M:].clone()
    q = Linear(io_dtype=pkg.scan._DTYPES[dtype], T=T, M=M, K=K, x_pitch=pitch, y_pitch=M + 8, x=x.data_ptr(), weight=w.data_ptr(), y=y.data_ptr(), residual=y.data_ptr(),
               weight_kxm=1, accumulate=1)
    L.check(lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)), "mpa_linear_run")
    assert rel_err(y[:, :M].float(), want) <= TOL[dtype] and torch.equal(y[:, M:], pad)


# widths that 16-byte rows do not divide, beside one that they do
@pytest.mark.parametrize("width", [12, 16, 18])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_stack_of_any_width(pkg, dev, width, dtype):
    torch.manual_seed(width)
    cfg = dict(d_model=width, n_layers=2, expand_factor=2)
    ref = pkg.Mamba(pkg.MambaConfig(**cfg)).to(dev)
    m = pkg.Mamba(pkg.MambaConfig(**cfg)).to(dev)
    m.load_state_dict(ref.state_dict())
    m = m.to(dtype)
    ref.load_state_dict(m.state_dict())
    x = torch.randn(2, 37, width, device=dev).to(dtype)
    want = ref(x.float())
    want.sum().backward()
    with torch.no_grad():
        assert rel_err(m(x).float(), want) <= 2 * TOL[dtype]
    y = m(x)
    y.sum().backward()
    assert rel_err(y.float(), want) <= 2 * TOL[dtype]
    a, b = (t.layers[0].mixer.in_proj.weight.grad.float() for t in (m, ref))
    assert rel_err(a, b) <= 5 * TOL[dtype]


# float32 x, y and residual around a bfloat16 product, over the tiles of the dispatch and their remainders
@pytest.mark.parametrize("T,M,K,pitch", [(1, 4, 8, 8), (33, 100, 72, 80), (65, 520, 1032, 1032), (500, 1540, 264, 264), (700, 1000, 1096, 1096),
                                         (1000, 1288, 64, 128), (2047, 900, 136, 144)])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_linear_with_a_float32_residual_stream(pkg, dev, T, M, K, pitch, accumulate):
    L, lib = pkg._lib, pkg._lib.load()
    g = torch.Generator().manual_seed(T)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev)
    x, w, bias, res, nw = rand(T, pitch), rand(M, K).bfloat16(), rand(M).bfloat16(), rand(T, M), rand(K)
    ssq, eps = rand(5, T).square() * K / 5, 1e-5
    normed = (x[:, :K].double() * (ssq.double().sum(0) / K + eps).rsqrt()[:, None] * nw.double()).bfloat16().double()
    want = normed @ w.double().t() + bias.double()
    X, Y, R = 256, 512, 1024

    def run(flags, x, y, res, y_ssq=None, norm=True):
        q = Linear(io_dtype=1 | flags, T=T, M=M, K=K, x_pitch=x.stride(0), y_pitch=M, x=x.data_ptr(), weight=w.data_ptr(), bias=bias.data_ptr(),
                   y=y.data_ptr(), residual=res.data_ptr() if res is not None else None, accumulate=accumulate)
        if norm:
            q.norm_weight, q.x_ssq, q.ssq_parts, q.eps = nw.data_ptr(), ssq.data_ptr(), 5, eps
        if y_ssq is not None:
            q.y_ssq = y_ssq.data_ptr()
        L.check(lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)), "mpa_linear_run")
        return y

    wide = lambda: torch.full((T, M), float("nan"), device=dev)
    narrow = lambda: wide().bfloat16()
    out_ssq = torch.empty((M + 31) // 32, T, device=dev)
    # float32 all round: only the sums are rounded (and a normalised element here and there the other way than `normed`:
    # a difference of 2^-8 in one of K factors)
    y = run(X | Y | R, x, wide(), res, out_ssq)
    assert rel_err(y, want + res.double()) <= 1e-3
    assert rel_err(out_ssq.sum(0), y.double().square().sum(1)) <= 1e-5
    # one flag at a time gives the same within the rounding of what is bfloat16 then
    assert rel_err(run(X | Y, x, wide(), res.bfloat16()), want + res.bfloat16().double()) <= 1e-3
    assert rel_err(run(X | R, x, narrow(), res), want + res.double()) <= TOL[torch.bfloat16]
    assert rel_err(run(X | Y, x, wide(), None), want) <= 1e-3
    x16 = x.bfloat16()
    plain = x16[:, :K].double() @ w.double().t() + bias.double()
    assert rel_err(run(Y | R, x16, wide(), res, norm=False), plain + res.double()) <= 1e-5
    q = Linear(io_dtype=1 | X, T=T, M=M, K=K, x_pitch=pitch, y_pitch=M, x=x.data_ptr(), weight=w.data_ptr(), y=y.data_ptr())
    assert lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)) == 3     # float32 x only to be normalised


# so many tiles that an XCD takes those of its own steps, and as many where W is the larger operand
@pytest.mark.parametrize("T,M", [(4111, 1288), (1288, 4112)])
@pytest.mark.parametrize("kxm", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_of_many_tiles(pkg, dev, T, M, kxm, dtype):
    L, lib, K = pkg._lib, pkg._lib.load(), 72
    g = torch.Generator().manual_seed(T)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev).to(dtype)
    x, w = rand(T, K), rand(K, M) if kxm else rand(M, K)
    y = torch.full((T, M), float("nan"), device=dev, dtype=dtype)
    q = Linear(io_dtype=pkg.scan._DTYPES[dtype], T=T, M=M, K=K, x_pitch=K, y_pitch=M, x=x.data_ptr(), weight=w.data_ptr(), y=y.data_ptr(),
               weight_kxm=kxm)
    L.check(lib.mpa_linear_run(ctypes.byref(q), pkg.scan._stream(dev)), "mpa_linear_run")
    want = x.double() @ (w.double() if kxm else w.double().t())
    assert rel_err(y, want) <= (1e-5 if dtype == torch.float32 else 2.0 ** -8)      # 72 products in float32; rounded once
