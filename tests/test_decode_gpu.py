"""The decode kernels (csrc/decode.hip) against the float64 layer: one token through a stack of
residual blocks, at the edges of their tiles (16 rows, 16 sequences, the K chunks), with odd low-rank
widths and every tap count, and the shapes they leave to the composed path."""
import pytest
import torch
import torch.nn.functional as F

from oracle import scan_oracle as so
from util import TOL, rel_err

pytestmark = pytest.mark.gpu


def layer_step_ref(layer, x, h, win):
    """float64 ResidualBlock.step (mambapy/mamba.py:114-125, 351-414) without the residual add at its end."""
    m, f64 = layer.mixer, lambda p: None if p is None else p.detach().double().cpu()
    cfg = m.config
    u = so.rmsnorm_ref(x, f64(layer.norm.weight), cfg.rms_norm_eps)
    xin, z = F.linear(u, f64(m.in_proj.weight), f64(m.in_proj.bias)).chunk(2, dim=1)
    full = torch.cat([win, xin.unsqueeze(2)], 2)
    xs = F.silu((full * f64(m.conv1d.weight)[:, 0]).sum(-1) + f64(m.conv1d.bias))
    dlow, B, C = F.linear(xs, f64(m.x_proj.weight)).split([cfg.dt_rank, cfg.d_state, cfg.d_state], dim=1)
    delta = so.softplus_ref(F.linear(dlow, f64(m.dt_proj.weight), f64(m.dt_proj.bias)))
    A = -torch.exp(f64(m.A_log))
    h = torch.exp(delta.unsqueeze(-1) * A) * h + (delta * xs).unsqueeze(-1) * B.unsqueeze(1)
    y = ((h * C.unsqueeze(1)).sum(-1) + f64(m.D) * xs) * F.silu(z)
    return F.linear(y, f64(m.out_proj.weight), f64(m.out_proj.bias)), h, full[:, :, 1:]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,width,kw", [
    (1, 8, {}), (1, 768, {}), (3, 264, {}),                       # smallest; a model's; dt_rank 17, ragged chunks
    (16, 72, dict(d_conv=2)), (17, 72, dict(d_conv=3)),           # one full tile of sequences, one more
    (33, 40, dict(d_state=4, expand_factor=1)),                   # 40 channels: the last row tile is half empty
    (64, 136, dict(d_state=20, dt_rank=5, bias=True)), (65, 64, dict(d_state=64)),
    (128, 1288, dict(d_state=8)),                                 # several batch tiles per workgroup
    (16, 520, dict(d_state=32, dt_rank=200)), (16, 1032, {}),     # x_proj within in_proj: most rows; not any more
    (129, 64, {}), (2, 64, dict(d_state=6)), (2, 64, dict(d_conv=5)),   # not taken by the kernels
])
def test_stack_step_matches_float64_layers(pkg, dev, dtype, batch, width, kw):
    torch.manual_seed(batch * 1000 + width)
    cfg = pkg.MambaConfig(d_model=width, n_layers=2, **kw)
    model = pkg.Mamba(cfg).to(dev).to(dtype)
    with torch.no_grad():
        for layer in model.layers:
            layer.norm.weight.uniform_(0.5, 1.5)
    cast = lambda t: t.to(dtype).to(dev)
    x = cast(torch.randn(batch, width))
    caches = [(torch.randn(batch, cfg.d_inner, cfg.d_state, device=dev), cast(torch.randn(batch, cfg.d_inner, cfg.d_conv - 1)))
              for _ in model.layers]
    caches[1] = (None, caches[1][1])        # zero state
    want = []
    xr = x.double().cpu()
    for layer, (h, w) in zip(model.layers, caches):
        h = torch.zeros(batch, cfg.d_inner, cfg.d_state).double() if h is None else h.double().cpu()
        y, h, w = layer_step_ref(layer, xr, h, w.double().cpu())
        xr = xr + y
        want.append((h, w))
    with torch.no_grad():
        before = [(h if h is None else h.clone(), w.clone()) for h, w in caches]
        y, new = model.step(x, list(caches))
        for (h, w), (h0, w0) in zip(caches, before):     # the old caches stay valid
            assert torch.equal(w, w0) and (h is None or torch.equal(h, h0))
        tol = TOL[dtype]
        assert rel_err(y, xr) <= tol
        for (h, w), (hr, wr) in zip(new, want):
            assert rel_err(h, hr) <= tol and rel_err(w, wr) <= tol
        own = [(torch.zeros_like(new[i][0]) if h is None else h.clone(), w.clone()) for i, (h, w) in enumerate(caches)]
        y2 = model.step_(x, own)                         # in place: the same kernels, the same results
        assert torch.equal(y2, y)
        assert all(torch.equal(a, b) for p, q in zip(own, new) for a, b in zip(p, q))


class Composed:
    """Stands in for the native layer code and takes no call: layers run module by module in Python."""
    block_train = block_step = stack_step = stack_forward = staticmethod(lambda *_: None)


def test_layer_handle_follows_its_module(pkg, dev, monkeypatch):
    """Weights changed in place or replaced, hooks, deep copies and conversions are all seen by the next call."""
    import copy
    torch.manual_seed(3)
    model = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev)
    x = torch.randn(2, 64, device=dev)
    seq = torch.randn(2, 9, 64, device=dev)

    def both(m):
        with torch.no_grad():
            return m.step(x.to(m.layers[0].mixer.D.dtype), m.empty_caches(2))[0], m(seq.to(m.layers[0].mixer.D.dtype))

    def composed(m):
        with monkeypatch.context() as mp:
            mp.setattr(pkg.modules, "_host", lambda: Composed)
            fresh = copy.deepcopy(m)        # (without the forms that the composed path keeps)
            for mod in fresh.modules():
                mod.__dict__.pop("_f32_cache", None)
            return both(fresh)

    def as_composed(m, step, forward):
        return all(rel_err(got, want) <= 1e-5 for got, want in zip((step, forward), composed(m)))

    a, fa = both(model)
    assert as_composed(model, a, fa)
    twin = copy.deepcopy(model)
    with torch.no_grad():
        model.layers[0].mixer.A_log.add_(0.5)
        model.layers[1].norm.weight.mul_(2.0)
        model.layers[1].mixer.out_proj.weight = torch.nn.Parameter(model.layers[1].mixer.out_proj.weight * 3)
    b, fb = both(model)
    assert as_composed(model, b, fb) and rel_err(b, a) > 1e-2
    c, fc = both(twin)
    assert torch.equal(c, a) and torch.equal(fc, fa)
    seen = []
    hook = model.layers[0].mixer.in_proj.register_forward_hook(lambda *_: seen.append(1))
    d, fd = both(model)
    assert len(seen) == 2 and rel_err(d, b) <= 1e-5 and rel_err(fd, fb) <= 1e-5
    hook.remove()
    half = model.to(torch.bfloat16)
    e, fe = both(half)
    assert rel_err(e, b) <= 3e-2 and rel_err(fe, fb) <= 3e-2
