"""Which products of many rows go to the package's own kernel (csrc/gemm_wide.hip: mpa_gemm_faster): the rule by itself, no GPU needed."""
import ctypes

import pytest


def taken(pkg, T, M, K, kxm=0):
    L = pkg._lib
    s = L.Gemm(x=256, weight=256, y=256, T=T, M=M, K=K, x_pitch=K, weight_pitch=M if kxm else K, y_pitch=M, weight_kxm=kxm)
    return L.load().mpa_gemm_faster(ctypes.byref(s)) == 1


# 1.04 to 1.42 times the library's time
@pytest.mark.parametrize("T,M,K,kxm", [
    (8000, 4096, 64, 0), (8000, 4096, 64, 1), (8000, 4096, 384, 0), (2048, 16384, 64, 0), (2048, 16384, 256, 0), (16384, 2048, 64, 1), (300, 128000, 64, 0), (300, 64000, 64, 0),
    (2048, 32768, 3080, 0), (6144, 16384, 3080, 0), (8000, 2048, 584, 0), (4000, 4096, 584, 0), (4000, 32000, 3080, 0), (8000, 32000, 584, 0),
    (4000, 64008, 640, 0), (300, 64008, 1536, 0), (4000, 128000, 584, 0),
])
def test_the_library_keeps_what_it_is_faster_at(pkg, T, M, K, kxm):
    assert not taken(pkg, T, M, K, kxm)


# 0.4 to 0.96
@pytest.mark.parametrize("width,T", [(256, 32000), (512, 8192), (392, 8000), (456, 10000), (680, 23200), (728, 4000)])
def test_layers_are_taken(pkg, width, T):
    assert taken(pkg, T, 4 * width, width)


@pytest.mark.parametrize("width,T", [(256, 64), (456, 10000), (600, 4000), (712, 2000), (712, 4000)])
def test_heads_are_taken(pkg, width, T):
    assert taken(pkg, T, 50280, width)
