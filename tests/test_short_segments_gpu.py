"""Backward scan of short sequences in segments of three to five tiles: at the lengths and workgroup counts where the cut begins, against the float64
oracle, and with gate, softplus and an initial state against the call that is not cut."""
import pytest
import torch

from oracle import c_oracle, scan_oracle as so
from util import GRAD_KEYS, TOL, rel_err, run_gpu_fwd_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Bs,L,ED,N,kw", [
    (1, 432, 64, 16, {}), (1, 433, 64, 16, {}), (3, 450, 70, 16, dict(reverse=True)), (85, 448, 40, 9, {}),  # 27 to 29 tiles: whole
    (1, 496, 64, 16, {}), (1, 497, 64, 16, {}),                        # 31 tiles: whole; 32, the last of one step
    (3, 520, 70, 16, dict(reverse=True)), (85, 500, 40, 9, {}),        # 33; 85 workgroups: three segments
    (86, 368, 33, 16, {}), (86, 369, 33, 16, dict(reverse=True)), (128, 393, 64, 16, {}),
    (86, 432, 33, 16, {}), (86, 433, 33, 16, dict(reverse=True)), (128, 450, 64, 16, {}),  # 86 and 128: two, from 28 tiles on
    (129, 393, 20, 16, {}),                                            # 129: not this cut
    (2, 208, 90, 24, {}), (2, 209, 90, 24, dict(reverse=True)), (2, 241, 90, 24, dict(reverse=True)),  # two passes over the states: from sixteen tiles on
    (2, 96, 65, 64, {}), (2, 97, 65, 64, {}), (2, 113, 65, 64, {}),    # four: from eight
    (2, 96, 33, 80, {}), (2, 97, 33, 80, {}), (1, 250, 10, 130, {}),   # five: from seven; two launches of the carry pass and more
    (1, 3100, 20, 16, {}), (1, 2999, 64, 40, dict(reverse=True)),      # 64 segments, of four tiles and one that is shorter
])
def test_against_oracle(pkg, dev, Bs, L, ED, N, kw):
    inp = so.make_inputs(Bs, L, ED, N, seed=Bs + L)
    flip = (lambda t: t.flip(1) if t.dim() == 3 else t) if kw else (lambda t: t)
    ref = c_oracle.sscan_fwd_bwd(**{k: flip(v) for k, v in inp.items()})
    got = run_gpu_fwd_bwd(pkg, inp, dev, **kw)
    for k in ("y",) + GRAD_KEYS:
        r = flip(ref[k]) if k not in ("dA", "dD") else ref[k]
        assert rel_err(got[k], r) <= TOL[torch.float32], k


@pytest.mark.parametrize("Bs,L,ED,N,dtype,reverse", [(2, 460, 100, 16, torch.bfloat16, False), (2, 560, 100, 16, torch.bfloat16, False), (1, 137, 1500, 48, torch.float32, True),
                                                     (5, 300, 250, 32, torch.bfloat16, True), (60, 400, 100, 16, torch.float32, False)])
def test_gated_against_uncut(pkg, dev, Bs, L, ED, N, dtype, reverse):
    g = torch.Generator().manual_seed(Bs)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev)
    base = dict(x=rand(Bs, L, ED).to(dtype), delta=(0.3 * rand(Bs, L, ED)).to(dtype), A=-torch.rand(ED, N, generator=g).to(dev) * 4 - 0.1,
                B=rand(Bs, L, N).to(dtype), C=rand(Bs, L, N).to(dtype), D=rand(ED), z=rand(Bs, L, ED).to(dtype), delta_bias=rand(ED) - 3,
                h0=rand(Bs, ED, N))
    base["x"] = base["x"].transpose(1, 2).contiguous().transpose(1, 2)  # (time fastest)
    dy, out = rand(Bs, L, ED).to(dtype), []
    for segments in (1, None):  # not cut; by the rule
        leaves = {k: v.clone().requires_grad_(k != "h0") for k, v in base.items()}
        with pkg.scan.plan_override(bwd_segments=segments):
            pkg.selective_scan_fn(**leaves, delta_softplus=True, reverse=reverse).backward(dy)
        out.append({k: v.grad for k, v in leaves.items() if k != "h0"})
    for k in out[0]:
        assert torch.isfinite(out[1][k]).all() and rel_err(out[1][k], out[0][k]) <= TOL[dtype], k
