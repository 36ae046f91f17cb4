"""RMSNorm on the gfx950 kernel: y = x * rsqrt(mean(x^2, -1) + eps) [* weight]
(mambapy/mamba.py:416-433), one pass forward and one backward instead of five elementwise
kernels each way."""
import torch

from . import _lib


def rmsnorm_supported(x) -> bool:
    """Shapes the kernel takes: float32 / bfloat16, last dim a multiple of 4 / 8 and at most
    2048 / 4096."""
    if x.dtype == torch.float32:
        return x.shape[-1] % 4 == 0 and x.shape[-1] <= 2048
    if x.dtype == torch.bfloat16:
        return x.shape[-1] % 8 == 0 and x.shape[-1] <= 4096
    return False


class RMSNormFn:
    @staticmethod
    def apply(x, weight, eps):
        return rmsnorm_fn(x, weight, eps)


class AddRMSNormFn:
    """(x, residual) -> (rmsnorm(x + residual), x + residual) in one pass each way."""

    @staticmethod
    def apply(x, residual, weight, eps):
        return add_rmsnorm_fn(x, residual, weight, eps)


def add_rmsnorm_fn(x, residual, weight=None, eps: float = 1e-5):
    """The residual add of the layer stack folded into the norm that reads its result
    (mambapy/mamba.py:106-112).  Returns (rmsnorm(x + residual) [* weight], x + residual)."""
    return _lib.host().rmsnorm(x, residual, weight, float(eps))


def rmsnorm_fn(x, weight=None, eps: float = 1e-5):
    """x : (..., d);  weight : (d) or None.  Returns a contiguous tensor of x's shape."""
    return _lib.host().rmsnorm(x, None, weight, float(eps))[0]
