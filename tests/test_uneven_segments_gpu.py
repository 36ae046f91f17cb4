"""Backward scan with more than half of the CUs covered, but not all: sequences cut in two parts of different lengths, at the workgroup counts and
lengths where the cut begins and ends, against the float64 oracle, and with gate and softplus against the call that is not cut."""
import pytest
import torch

from oracle import c_oracle, scan_oracle as so
from util import GRAD_KEYS, TOL, rel_err, run_gpu_fwd_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Bs,L,ED,N,kw", [
    (43, 401, 150, 16, {}),                              # 129 workgroups, the shortest that is cut
    (43, 384, 150, 16, {}),                              # a tile fewer: not cut
    (160, 433, 40, 16, dict(reverse=True)),              # 160: two short parts in turn
    (161, 560, 33, 12, {}), (192, 577, 64, 16, {}),      # 161, 192: three
    (193, 1205, 20, 16, {}), (224, 1216, 9, 24, dict(reverse=True)),  # 193, 224: seven; two passes over the states
    (225, 1216, 9, 16, {}),                              # 225: not cut
])
def test_against_oracle(pkg, dev, Bs, L, ED, N, kw):
    inp = so.make_inputs(Bs, L, ED, N, seed=Bs + L)
    flip = (lambda t: t.flip(1) if t.dim() == 3 else t) if kw else (lambda t: t)
    ref = c_oracle.sscan_fwd_bwd(**{k: flip(v) for k, v in inp.items()})
    got = run_gpu_fwd_bwd(pkg, inp, dev, **kw)
    for k in ("y",) + GRAD_KEYS:
        r = flip(ref[k]) if k not in ("dA", "dD") else ref[k]
        assert rel_err(got[k], r) <= TOL[torch.float32], k


@pytest.mark.parametrize("Bs,L,ED,N,dtype", [(150, 450, 30, 16, torch.bfloat16), (64, 600, 190, 16, torch.float32), (200, 1300, 24, 32, torch.bfloat16)])
def test_gated_against_uncut(pkg, dev, Bs, L, ED, N, dtype):
    g = torch.Generator().manual_seed(Bs)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev)
    base = dict(x=rand(Bs, L, ED).to(dtype), delta=(0.3 * rand(Bs, L, ED)).to(dtype), A=-torch.rand(ED, N, generator=g).to(dev) * 4 - 0.1,
                B=rand(Bs, L, N).to(dtype), C=rand(Bs, L, N).to(dtype), D=rand(ED), z=rand(Bs, L, ED).to(dtype), delta_bias=rand(ED) - 3,
                h0=rand(Bs, ED, N))
    dy, out = rand(Bs, L, ED).to(dtype), []
    for segments in (1, None):  # not cut; by the rule
        leaves = {k: v.clone().requires_grad_(k != "h0") for k, v in base.items()}
        with pkg.scan.plan_override(bwd_segments=segments):
            pkg.selective_scan_fn(**leaves, delta_softplus=True).backward(dy)
        out.append({k: v.grad for k, v in leaves.items() if k != "h0"})
    for k in out[0]:
        assert torch.isfinite(out[1][k]).all() and rel_err(out[1][k], out[0][k]) <= TOL[dtype], k
