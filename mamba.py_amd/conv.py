"""Causal depthwise convolution along time (+ bias, + SiLU) on the gfx950 kernel.

`causal_conv1d_fn(x, weight, bias)` is what MambaBlock.forward computes with
    conv1d(x.transpose(1, 2))[:, :, :L].transpose(1, 2) followed by silu
(mambapy/mamba.py:217-221), on the (B, L, ED) tensor directly: any strides are read in place,
the result is a new (B, L, ED) tensor with unit stride along ED.
"""
from . import _lib
from .scan import _io_dtype


def _conv_shape(x, y_like, g_like, K, silu):
    s = _lib.ConvShape()
    s.batch, s.seqlen, s.dim = x.shape
    s.kernel = K
    s.io_dtype = _io_dtype(x)
    s.flags = _lib.MPA_CONV_SILU if silu else 0
    s.x_sb, s.x_sl, s.x_sd = x.stride()
    s.y_sb, s.y_sl, s.y_sd = y_like.stride()
    s.g_sb, s.g_sl, s.g_sd = g_like.stride()
    return s


class CausalConv1dFn:
    @staticmethod
    def apply(x, weight, bias=None, window=None, silu=True, return_window=False):
        return causal_conv1d_fn(x, weight, bias, window, silu, return_window)


def causal_conv1d_update(x, window, weight, bias=None, silu=True):
    """One decode step of the convolution (mambapy/mamba.py:366-369, 379) in one kernel:
    x : (B, ED) newest input (any row stride);  window : (B, ED, K-1) contiguous rolling cache of
    the previous inputs, UPDATED IN PLACE (oldest dropped, x appended).  Returns
    silu(conv) as (B, ED).  No autograd: decoding runs under torch.no_grad()."""
    return _lib.host().conv_update(x, window, weight, bias, bool(silu))


def causal_conv1d_fn(x, weight, bias=None, window=None, silu=True, return_window=False):
    """x : (B, L, ED) (any strides);  weight : (ED, 1, K) or (ED, K), K in 2..4;  bias : (ED).
    window : optional (B, ED, K-1) inputs before step 0 (zeros if None).
    Returns silu(conv(x)) as (B, L, ED) [, the last K-1 inputs as (B, ED, K-1)]."""
    y, wout = _lib.host().conv(x, weight, bias, window, bool(silu), bool(return_window))
    return (y, wout) if return_window else y
