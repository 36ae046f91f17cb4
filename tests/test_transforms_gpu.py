"""Derivatives that the package has no rule for are refused, never dropped: forward mode and functorch's transforms, for
the operators and for layers on their native path, in inputs and in parameters."""
import pytest
import torch
import torch.autograd.forward_ad as fwd

pytestmark = pytest.mark.gpu


def operators(pkg, dev):
    torch.manual_seed(1)
    Bs, L, ED, N = 2, 20, 64, 16
    r = lambda *s: torch.randn(*s, device=dev)
    A = -torch.rand(ED, N, device=dev) - 0.1
    return {
        "scan": (pkg.selective_scan_fn, [r(Bs, L, ED), r(Bs, L, ED).exp(), A, r(Bs, L, N), r(Bs, L, N), r(ED)]),
        "pscan": (pkg.pscan, [torch.rand(Bs, L, ED, N, device=dev), r(Bs, L, ED, N)]),
        "conv": (pkg.causal_conv1d_fn, [r(Bs, L, ED), r(ED, 4), r(ED)]),
        "norm": (pkg.rmsnorm_fn, [r(Bs, L, ED), r(ED)]),
        "add_norm": (pkg.add_rmsnorm_fn, [r(Bs, L, ED), r(Bs, L, ED), r(ED)]),
    }


@pytest.mark.parametrize("name", ["scan", "pscan", "conv", "norm", "add_norm"])
def test_operators_refuse(pkg, dev, name):
    fn, args = operators(pkg, dev)[name]
    for i in range(len(args)):
        with fwd.dual_level():
            dual = list(args)
            dual[i] = fwd.make_dual(args[i], torch.ones_like(args[i]))
            with pytest.raises(NotImplementedError):
                fn(*dual)
            with torch.no_grad(), pytest.raises(NotImplementedError):
                fn(*dual)
        rest = lambda t: fn(*args[:i], t, *args[i + 1:])
        first = lambda t: rest(t) if torch.is_tensor(rest(t)) else rest(t)[0]
        with pytest.raises(RuntimeError):
            torch.func.vmap(rest)(torch.stack([args[i]] * 2))
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: first(t).sum())(args[i])
        with pytest.raises(RuntimeError):
            torch.func.jvp(first, (args[i],), (torch.ones_like(args[i]),))
    with fwd.dual_level():      # a level without tangents is no reason
        fn(*args)
    fn(*args)


def test_layers_refuse(pkg, dev):
    torch.manual_seed(2)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev)
    blk = m.layers[0].mixer
    x = torch.randn(2, 20, 64, device=dev)

    def runs(x, m):
        yield lambda: m.layers[0].mixer(x)
        yield lambda: m(x)
        with torch.no_grad():
            yield lambda: m.layers[0].mixer(x)
            yield lambda: m(x)
            yield lambda: m.step(x[:, 0], m.empty_caches(2))

    for run in runs(x, m):
        want = run()
        with fwd.dual_level():
            got = run()
        a, b = (r[0] if isinstance(r, tuple) else r for r in (got, want))
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)
    with fwd.dual_level():
        for run in runs(fwd.make_dual(x, torch.ones_like(x)), m):
            with pytest.raises(NotImplementedError):
                run()
        for name in ("A_log", "D", "conv1d.weight", "conv1d.bias", "in_proj.weight", "x_proj.weight"):
            p = dict(blk.named_parameters())[name]
            swapped = {name: fwd.make_dual(p.detach(), torch.ones_like(p))}
            for mode in (torch.enable_grad, torch.no_grad):
                with mode(), pytest.raises(NotImplementedError):
                    torch.func.functional_call(blk, swapped, (x,))
    with pytest.raises(RuntimeError):
        torch.func.vmap(m)(torch.stack([x, x]))
    with torch.no_grad(), pytest.raises(RuntimeError):
        torch.func.vmap(m)(torch.stack([x, x]))
