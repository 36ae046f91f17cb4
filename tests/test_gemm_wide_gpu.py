"""Products of many rows by 256 x 256 tiles (csrc/gemm_wide.hip): ends of T, M and K within tiles, halves of tiles and stages, fewer stages than are
in flight, one to three rounds with and without halves, pitches, both forms of the weight; rows and columns around the operands hold NaN."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kxm", [0, 1])
@pytest.mark.parametrize("T,M,K,pad", [
    (1, 8, 8, 0), (129, 264, 64, 8), (255, 248, 72, 0), (256, 256, 128, 8), (300, 520, 136, 0), (700, 264, 200, 24), (1000, 1000, 776, 8),
    (2048, 2048, 192, 0),                            # 64 tiles, as halves
    (8000, 1536, 264, 8), (8191, 2040, 328, 0),      # one round of whole tiles, the last a row and eight columns short
    (8193, 2056, 64, 8),                             # one round and halves, of which some are beyond T
    (24000, 1536, 128, 0), (16500, 3080, 520, 8),    # two rounds and halves in one round and in two
])
def test_against_float64(pkg, dev, T, M, K, pad, kxm):
    L = pkg._lib
    lib = L.load()
    g = torch.Generator(device=dev).manual_seed(T + M + K)
    rand = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()

    def within(rows, cols):
        t = torch.full((rows + 3, cols + pad), float("nan"), dtype=torch.bfloat16, device=dev)
        t[:rows, :cols] = rand(rows, cols)
        return t[:rows, :cols]
    x, w = within(T, K), within(*((K, M) if kxm else (M, K)))
    y = torch.full((T + 1, M + pad), -7.0, dtype=torch.bfloat16, device=dev)
    s = L.Gemm(x=x.data_ptr(), weight=w.data_ptr(), y=y.data_ptr(), T=T, M=M, K=K, x_pitch=K + pad, weight_pitch=w.stride(0), y_pitch=M + pad, weight_kxm=kxm)
    L.check(lib.mpa_gemm_run(ctypes.byref(s), pkg.scan._stream(dev)), "mpa_gemm_run")
    wd = w.double() if kxm else w.double().t()
    bad = 0
    for t0 in range(0, T, 4096):
        xd, got = x[t0:t0 + 4096].double(), y[t0:min(t0 + 4096, T), :M].double()
        want, size = xd @ wd, xd.abs() @ wd.abs()
        # float32 sums: K roundings of 2^-24 of the sum of magnitudes at most; a result is rounded once
        bad += (~((got - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * size)).sum().item()
    assert bad == 0
    assert (y[T:] == -7).all() and (y[:, M:] == -7).all()


def test_refuses(pkg, dev):
    L = pkg._lib
    lib = L.load()
    t = torch.zeros(64, 64, dtype=torch.bfloat16, device=dev)
    good = dict(x=t.data_ptr(), weight=t.data_ptr(), y=t.data_ptr(), T=8, M=8, K=8, x_pitch=8, weight_pitch=8, y_pitch=8)
    for change in (dict(x=None), dict(M=12), dict(K=4), dict(T=0), dict(x_pitch=4), dict(y_pitch=12), dict(weight=t.data_ptr() + 2), dict(x_pitch=1 << 23)):
        s = L.Gemm(**{**good, **change})
        assert lib.mpa_gemm_run(ctypes.byref(s), pkg.scan._stream(dev)) != 0 and lib.mpa_gemm_faster(ctypes.byref(s)) == 0


@pytest.mark.parametrize("T,M,K,kxm,faster", [
    (24000, 3072, 768, 0, 1), (24000, 1536, 1536, 0, 0), (8000, 3072, 768, 0, 1), (16384, 3072, 768, 0, 0), (8192, 2048, 512, 0, 1),
    (4000, 2912, 728, 0, 1), (1700, 728, 1456, 0, 0), (8000, 768, 3072, 1, 0), (7000, 728, 2912, 1, 1), (8000, 50280, 768, 0, 0),
])
def test_rule(pkg, dev, T, M, K, kxm, faster):
    L = pkg._lib
    s = L.Gemm(x=256, weight=256, y=256, T=T, M=M, K=K, x_pitch=K, weight_pitch=M if kxm else K, y_pitch=M, weight_kxm=kxm)
    assert L.load().mpa_gemm_faster(ctypes.byref(s)) == faster
