"""Weight gradients by 256 x 256 tiles (csrc/wgrad_wide.hip): remainders of T around its stages, of rows and columns around whole and narrow tiles on
either side, kept columns, gaps, strides, and rows beyond the last that hold NaN."""
import ctypes

import pytest
import torch

from test_wgrad_plan import small_tile_bytes

pytestmark = pytest.mark.gpu


SIZES = [
    # (columns of P, of Q, kept columns, first row of the gap, gap)
    (8000, [(3072, 768, 768, 0, 0), (768, 1536, 1536, 0, 0), (96, 1536, 1536, 48, 16), (1536, 64, 48, 0, 0)]),
    (8161, [(3080, 776, 776, 0, 0), (904, 1672, 1665, 0, 0), (136, 1544, 1544, 0, 0), (1544, 72, 71, 1536, 8)]),  # rests of 8, 136, 128 + 8
    (16385, [(2176, 1152, 1152, 0, 0), (384, 2176, 2176, 255, 3), (128, 8, 8, 0, 0), (8, 2048, 2048, 0, 0)]),      # rests of 128
    (4127, [(4096, 1024, 1024, 0, 0), (1024, 2048, 2048, 0, 0), (256, 2056, 2051, 0, 0), (2056, 256, 255, 100, 300)]),
    (1500, [(8192, 2048, 2048, 0, 0), (2048, 4096, 4096, 0, 0)]),  # (one part of T and whole tiles: both kernels ask for the same workspace)
]


@pytest.mark.parametrize("T,sizes", SIZES)
def test_against_float64_products(pkg, dev, T, sizes):
    L = pkg._lib
    lib = L.load()
    g = torch.Generator(device=dev).manual_seed(T)
    jobs, hold = (L.WgradJob * len(sizes))(), []
    for j, (M, N, kept, at, gap) in zip(jobs, sizes):
        def rows(cols, pad):
            t = torch.full((T + 33, cols + pad), float("nan"), dtype=torch.bfloat16, device=dev)
            t[:T, 8:8 + cols] = torch.randn(T, cols, generator=g, device=dev).bfloat16()
            return t[:T, 8:8 + cols]
        P, Q = rows(M, 16), rows(N, 24)
        out = torch.full((M - gap, kept), float("nan"), dtype=torch.bfloat16, device=dev)
        j.p, j.q, j.ldp, j.ldq, j.out = P.data_ptr(), Q.data_ptr(), P.stride(0), Q.stride(0), out.data_ptr()
        j.rows, j.cols, j.keep_cols, j.gap_at, j.gap = M, N, kept, at, gap
        hold.append((P, Q, out, kept, at, gap))
    n = lib.mpa_wgrad_workspace_bytes(jobs, len(sizes), T, 1)
    # (the kernel of this file, and not the one of smaller tiles)
    assert n != small_tile_bytes(sizes, T) or all(s[0] % 256 == 0 and s[1] % 256 == 0 for s in sizes)
    ws = torch.full((n + 256,), 255, dtype=torch.uint8, device=dev)
    call = lambda size: lib.mpa_wgrad(jobs, len(sizes), T, 1, ctypes.c_void_p(ws.data_ptr()), size, pkg.scan._stream(dev))
    assert call(n - 1) == lib.mpa_wgrad(jobs, len(sizes), T, 1, ctypes.c_void_p(ws.data_ptr()), 0, pkg.scan._stream(dev)) != 0
    L.check(call(n), "mpa_wgrad")
    assert (ws[n:] == 255).all()
    for P, Q, out, kept, at, gap in hold:
        drop = lambda m: torch.cat([m[:at], m[at + gap:]])[:, :kept]
        p, q = P.double(), Q.double()
        want, size = drop(p.t() @ q), drop(p.abs().t() @ q.abs())
        # float32 sums (T roundings of 2^-24 of the sum of magnitudes at most, and of either sign: a root of T), rounded to bfloat16 once
        assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + T ** 0.5 * 2.0 ** -24 * size).all()
