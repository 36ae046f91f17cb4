"""Layers whose submodules, methods or hooks are not the plain ones: the native calls step aside, before and after they
have run on the model.  The yardstick is the same model module by module in Python."""
import copy
import types

import pytest
import torch
import torch.nn as nn
import torch.nn.utils.parametrize as parametrize
import torch.nn.utils.prune as prune

from util import rel_err

pytestmark = pytest.mark.gpu


class Nothing:
    """Stands in for the native layer code and takes no call."""
    block_train = block_step = stack_step = stack_forward = staticmethod(lambda *_: None)


def results(m, x):
    """Every way of running the stack: forward and step without gradients, forward and backward with."""
    with torch.no_grad():
        y, caches = m(x, return_caches=True)
        s, after = m.step(x[:, 0], list(caches))
        out = [y, s] + [t for pair in caches + after for t in pair]
        own = [(h.clone(), w.clone()) for h, w in caches]
        out.append(m.step_(x[:, 0], own))
        out.append(m.layers[1].mixer.step(x[:, 0], caches[1])[0])
    xr = x.clone().requires_grad_()
    y = m(xr)
    leaves = [xr] + [p for p in m.parameters() if p.requires_grad]
    return out + [y.detach()] + list(torch.autograd.grad(y, leaves, torch.ones_like(y)))


class Doubled(nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


class Raised(nn.Module):
    def forward(self, w):
        return w + 1


def half_of(module, name):
    p = getattr(module, name).requires_grad_(False)      # (pruning forms the value once, with its graph, and again in forward)
    prune.custom_from_mask(module, name, torch.arange(p.numel(), device=p.device).view_as(p) % 2)


def wrap_forward(m):
    lin = m.layers[0].mixer.in_proj
    inner = lin.forward
    lin.forward = lambda x: 2 * inner(x)


def wrap_ssm(m):
    b = m.layers[0].mixer
    inner = b.ssm
    b.ssm = lambda x, z=None, **kw: 0.5 * inner(x, z, **kw) if not kw.get("return_last_state") else (lambda r: (0.5 * r[0], r[1]))(inner(x, z, **kw))


def other_class(m):
    m.layers[1].mixer.out_proj.__class__ = Doubled


def other_D(m):
    m.layers[1].mixer._D = types.MethodType(lambda self: 2 * self.D, m.layers[1].mixer)


CHANGES = {
    "forward of a projection": wrap_forward,
    "class of a projection": other_class,
    "ssm of a block": wrap_ssm,
    "D of a block": other_D,
    "conv bias pruned": lambda m: half_of(m.layers[0].mixer.conv1d, "bias"),
    "dt bias pruned": lambda m: half_of(m.layers[0].mixer.dt_proj, "bias"),
    "norm weight pruned": lambda m: half_of(m.layers[0].norm, "weight"),
    "conv bias parametrised": lambda m: parametrize.register_parametrization(m.layers[0].mixer.conv1d, "bias", Raised()),
    "dt bias parametrised": lambda m: parametrize.register_parametrization(m.layers[1].mixer.dt_proj, "bias", Raised()),
    "norm weight parametrised": lambda m: parametrize.register_parametrization(m.layers[1].norm, "weight", Raised()),
    "hook of a norm": lambda m: m.layers[0].norm.register_forward_hook(lambda mod, args, out: 0.5 * out),
    "eps of a norm": lambda m: setattr(m.layers[1].norm, "eps", 0.5),
    "projection replaced": lambda m: setattr(m.layers[0].mixer, "in_proj", nn.Linear(64, 256, bias=True, device="cuda")),
}


@pytest.mark.parametrize("used_before", [False, True])
@pytest.mark.parametrize("change", CHANGES)
def test_what_a_module_was_given_is_used(pkg, dev, monkeypatch, change, used_before):
    torch.manual_seed(1)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev)
    x = torch.randn(2, 40, 64, device=dev)
    before = results(copy.deepcopy(m), x)
    if used_before:
        results(m, x)
    CHANGES[change](m)
    got = results(m, x)
    with monkeypatch.context() as mp:
        mp.setattr(pkg.modules, "_host", lambda: Nothing)
        want = results(m, x)
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        assert rel_err(a, b) <= 1e-4, i
    # the change is one that shows (outputs and states)
    assert max(rel_err(a, b) for a, b in zip(got[:6], before[:6])) > 1e-2


def test_methods_of_the_classes_are_used(pkg, dev, monkeypatch):
    torch.manual_seed(2)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev)
    x = torch.randn(2, 40, 64, device=dev)
    results(m, x)
    for cls, name in ((pkg.MambaBlock, "_D"), (pkg.RMSNorm, "_w"), (nn.Linear, "forward")):
        seen, inner = [], cls.__dict__[name]
        with monkeypatch.context() as mp:
            mp.setattr(cls, name, lambda self, *a: (seen.append(1), inner(self, *a))[1])
            results(m, x)
        # forward, step, step_ and training of two layers
        assert len(seen) >= 8, name


def test_global_hooks_see_the_submodules(pkg, dev):
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev)
    x = torch.randn(2, 40, 64, device=dev)
    results(m, x)
    seen = []
    hook = nn.modules.module.register_module_forward_hook(lambda mod, *_: seen.append(mod))
    try:
        m(x)
        with torch.no_grad():
            m(x)
            m.step(x[:, 0], m.empty_caches(2))
    finally:
        hook.remove()
    assert sum(mod is m.layers[0].mixer.in_proj for mod in seen) == 3


def test_options_are_read_in_every_call(pkg, dev, monkeypatch):
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev)
    x = torch.randn(2, 40, 64, device=dev)
    blk = m.layers[0].mixer
    assert blk(x).grad_fn.name() == "MambaBlockBackward"
    taken = []
    real = pkg.modules._host()
    spy = types.SimpleNamespace(**{n: (lambda *a, f=getattr(real, n): (lambda r: (taken.append(r is not None), r)[1])(f(*a)))
                                   for n in ("block_train", "stack_forward", "stack_step", "block_step")})
    monkeypatch.setattr(pkg.modules, "_host", lambda: spy)

    def run():
        taken.clear()
        blk(x)
        with torch.no_grad():
            m(x)
        return taken

    assert run() == [True, True]
    blk.config.fused_softplus = False
    assert run() == [False, False]
    blk.config.fused_softplus = True
    assert run() == [True, True]
    monkeypatch.setattr(pkg.modules, "PAD_PROJECTIONS", False)
    assert True not in run()
