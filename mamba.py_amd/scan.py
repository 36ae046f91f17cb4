"""Host side of the selective-scan hot path: the reference's operator surface
(`pscan`, `selective_scan`, `ssm_step`) bound to the gfx950 kernels through the C ABI.

Mirrors, by name and argument meaning:
  pscan(A, X)                                   mambapy/pscan.py:151-226
  selective_scan(x, delta, A, B, C, D)          mambapy/mamba.py:274-295
  selective_scan_fn(..., z=, delta_bias=, delta_softplus=)   the fused call of mamba.py:259-260
  ssm_step(x, delta, A, B, C, D, h)             mambapy/mamba.py:400-412
PyTorch supplies device memory, streams and the autograd graph; all arithmetic runs in
libmambapy_amd.so, called from csrc/host.cpp.  Tensors must live on a ROCm device: there is no CPU path.
"""
import contextlib
import ctypes
import os

import torch

from . import _lib

_DTYPES = {torch.float32: _lib.MPA_F32, torch.bfloat16: _lib.MPA_BF16}


def _io_dtype(t: torch.Tensor) -> int:
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}: the kernels take float32 or bfloat16 "
                        "tensors (state and accumulation are float32 in both cases)") from None


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream(device):
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


class LaunchPlan:
    """Overrides of the decomposition the library would choose from the shape (None / False =
    let it choose).  The library itself reads no environment: the MPA_* variables below are
    read here, once, when the module is imported, and travel to the kernels inside the shape
    struct of every call.

        MPA_FWD_NS / MPA_BWD_NS       states of d_state per lane (a power of two)
        MPA_FWD_NSEG / MPA_BWD_NSEG   segments a sequence is cut into (1 = never cut)
        MPA_PSCAN_CHUNKS              pieces the generic scan cuts a sequence into (1 = never cut)
        MPA_BWD_GENERAL=1             general backward kernel even where the fast one applies
        MPA_GROUP_CHANNELS            64, 48, 32 or 16 channels of a batch row per workgroup
    """
    _FIELDS = ("fwd_states_per_lane", "bwd_states_per_lane", "fwd_segments", "bwd_segments",
               "bwd_general", "expire_waits", "pscan_chunks", "group_channels")

    def __init__(self):
        env = lambda k: int(os.environ[k]) if os.environ.get(k, "").strip() else None
        self.fwd_states_per_lane = env("MPA_FWD_NS")
        self.bwd_states_per_lane = env("MPA_BWD_NS")
        self.fwd_segments = env("MPA_FWD_NSEG")
        self.bwd_segments = env("MPA_BWD_NSEG")
        self.pscan_chunks = env("MPA_PSCAN_CHUNKS")
        self.bwd_general = os.environ.get("MPA_BWD_GENERAL", "") == "1"
        self.expire_waits = False  # test hook (MPA_PLAN_EXPIRE_WAITS)
        self.group_channels = env("MPA_GROUP_CHANNELS")  # channels per workgroup (None: the library picks)
        self.__dict__["packed"] = self._pack()

    def __setattr__(self, name, value):
        self.__dict__[name] = value
        if len(self.__dict__) > len(self._FIELDS):      # not while __init__ is filling the fields in
            self.__dict__["packed"] = self._pack()

    def _pack(self):
        """The fields as csrc/host.cpp takes them (Plan)."""
        return (self.fwd_states_per_lane or 0, self.bwd_states_per_lane or 0, self.fwd_segments or 0, self.bwd_segments or 0,
                self._flags(), self.pscan_chunks or 0)

    def _flags(self):
        return (_lib.MPA_PLAN_BWD_GENERAL if self.bwd_general else 0) | \
               (_lib.MPA_PLAN_EXPIRE_WAITS if self.expire_waits else 0) | \
               {None: 0, 64: _lib.MPA_PLAN_GROUP_64, 48: _lib.MPA_PLAN_GROUP_48, 32: _lib.MPA_PLAN_GROUP_32,
                16: _lib.MPA_PLAN_GROUP_16}[self.group_channels]

    def fill(self, shape, backward):
        shape.plan_states_per_lane = (self.bwd_states_per_lane if backward else self.fwd_states_per_lane) or 0
        shape.plan_segments = (self.bwd_segments if backward else self.fwd_segments) or 0
        shape.plan_flags = self._flags()


plan = LaunchPlan()


@contextlib.contextmanager
def plan_override(**kw):
    """with plan_override(fwd_segments=4, bwd_states_per_lane=2): ...  (tuning and tests)"""
    for k in kw:
        if k not in LaunchPlan._FIELDS:
            raise TypeError(f"unknown plan field {k!r}")
    old = {k: getattr(plan, k) for k in kw}
    for k, v in kw.items():
        setattr(plan, k, v)
    try:
        yield plan
    finally:
        for k, v in old.items():
            setattr(plan, k, v)


def _sscan_shape(x, delta, Bm, y_like, g_like, dbc_like, N, flags, z=None, backward=False):
    """Shape struct of one call.  delta may be float32 next to bfloat16 tensors (the reference's call
    under autocast, mambapy/mamba.py:264-265): the library then reads it, and writes ddelta, as float32."""
    s = _lib.SscanShape()
    s.batch, s.seqlen, s.dim = x.shape
    s.dstate = N
    s.io_dtype = _io_dtype(x)
    s.flags = flags
    s.u_sb, s.u_sl, s.u_sd = x.stride()
    if z is not None:
        s.z_sb, s.z_sl, s.z_sd = z.stride()
    s.d_sb, s.d_sl, s.d_sd = delta.stride()
    s.delta_dtype = _lib.MPA_DELTA_F32 if (delta.dtype == torch.float32 and x.dtype != torch.float32) else 0
    s.y_sb, s.y_sl, s.y_sd = y_like.stride()
    s.g_sb, s.g_sl, s.g_sd = g_like.stride()
    s.bc_sb, s.bc_sl = Bm.stride(0), Bm.stride(1)
    s.dbc_sb, s.dbc_sl = dbc_like.stride(0), dbc_like.stride(1)
    plan.fill(s, backward)
    return s


class SelectiveScanFn:
    """Fused discretise -> scan -> readout with a hand-written backward kernel (the graph node is
    csrc/host.cpp: ScanBackward)."""

    @staticmethod
    def apply(x, delta, A, B, C, D, z=None, delta_bias=None, delta_softplus=False, h0=None, return_last_state=False,
              need_grad=None, reverse=False):
        """need_grad is decided from the grad mode and the inputs; False switches gradients off."""
        with contextlib.nullcontext() if need_grad is not False else torch.no_grad():
            return selective_scan_fn(x, delta, A, B, C, D, z, delta_bias, delta_softplus, h0, return_last_state, reverse)


def selective_scan_fn(x, delta, A, B, C, D, z=None, delta_bias=None, delta_softplus=False,
                      h0=None, return_last_state=False, reverse=False):
    """y = selective scan of (x, delta, A, B, C, D), optionally with softplus(delta + bias)
    and the gate y*silu(z) folded in (the fused form the reference reaches through
    `use_cuda`, mambapy/mamba.py:252-261), in this package's (B, L, ED) layout.

    x, delta, z : (B, L, ED);  A : (ED, N);  B, C : (B, L, N);  D, delta_bias : (ED);
    h0 : optional (B, ED, N) initial state.  Returns y (B, L, ED) [, last state (B, ED, N)].
    reverse=True runs the recurrence from the last step to the first: the same result as
    flipping x, delta, z, B, C along time, scanning and flipping y back (the backward direction
    of the reference's bidirectional block, mambapy/vim.py:228-261), without the copies; h0 is
    then the state before step L-1 and the last state the one after step 0.
    """
    y, h_last = _lib.host().scan(x, delta, A, B, C, D, z, delta_bias, bool(delta_softplus), h0,
                                 bool(return_last_state), bool(reverse), plan.packed)
    return (y, h_last) if return_last_state else y


def selective_scan(x, delta, A, B, C, D):
    """Drop-in for MambaBlock.selective_scan / selective_scan_seq
    (mambapy/mamba.py:274-327): same arguments, same result, differentiable."""
    return selective_scan_fn(x, delta, A, B, C, D)


# ------------------------------------------------------------------------------------------
# generic scan
# ------------------------------------------------------------------------------------------

class PScan:
    """H[t] = A[t]*H[t-1] + X[t] along dim 1 of (B, L, D, N) tensors; returns a new tensor
    and never modifies its inputs (mambapy/pscan.py:151-224).  Any L: no padding."""

    @staticmethod
    def apply(A_in, X_in, reverse=False):
        return _lib.host().pscan(A_in, X_in, bool(reverse), plan.packed)


pscan = PScan.apply


def pscan_rev(A, X):
    """H[t] = A[t]*H[t+1] + X[t], H[L] = 0: the scan of mambapy/pscan.py:94-149
    (PScan.pscan_rev, `flip . pscan . flip`) as a differentiable call of its own."""
    return PScan.apply(A, X, True)


# ------------------------------------------------------------------------------------------
# decode step
# ------------------------------------------------------------------------------------------

def ssm_step(x, delta, A, B, C, D, h=None, z=None, delta_bias=None, delta_softplus=False,
             inplace=False):
    """One token: h' = exp(delta*A)*h + delta*B*x, y = C.h' + D*x (mambapy/mamba.py:400-412).

    x, delta, z : (B, ED);  A : (ED, N);  B, C : (B, N);  D, delta_bias : (ED);
    h : (B, ED, N) float32 or None (zeros).  Returns (y, h').  By default h' is a new tensor
    and h is left untouched, as in the reference; inplace=True updates h itself.
    No autograd: decoding runs under torch.no_grad().
    """
    return _lib.host().step(x, delta, A, B, C, D, h, z, delta_bias, bool(delta_softplus), bool(inplace))
