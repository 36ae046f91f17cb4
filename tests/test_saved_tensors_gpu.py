"""What the graph nodes keep goes through torch's hooks on saved tensors: checkpointed and offloaded layers hold no
activations on the GPU, and their gradients are those of the plain pass, bit for bit."""
import pytest
import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

pytestmark = pytest.mark.gpu


def held_and_gradients(dev, forward, leaves, dy):
    """Bytes that live between the forward and the backward pass, beyond the output; the gradients."""
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(dev)
    y = forward()
    held = torch.cuda.memory_allocated(dev) - before - y.numel() * y.element_size()
    return held, torch.autograd.grad(y, leaves, dy)


@pytest.mark.parametrize("how", ["checkpoint", "save_on_cpu"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_blocks_give_their_activations_away(pkg, dev, dtype, how):
    torch.manual_seed(1)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=3)).to(dev).to(dtype)
    x = torch.randn(2, 600, 64, device=dev).to(dtype).requires_grad_()
    dy = torch.randn(2, 600, 64, device=dev).to(dtype)
    leaves = [x] + list(m.parameters())

    def through_layers():
        h = x
        for layer in m.layers:
            h = checkpoint(layer, h, use_reentrant=False)
        return h

    def offloaded():
        with torch.autograd.graph.save_on_cpu():
            return m(x)

    def plain():
        h = x
        for layer in m.layers:
            h = layer(h)
        return h

    if how == "checkpoint":
        held, got = held_and_gradients(dev, through_layers, leaves, dy)
        full, want = held_and_gradients(dev, plain, leaves, dy)
    else:
        held, got = held_and_gradients(dev, offloaded, leaves, dy)
        full, want = held_and_gradients(dev, lambda: m(x), leaves, dy)
    # a layer's activations are some twenty times its input; a checkpointed one keeps that input
    assert held <= 0.15 * full, (held, full)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("last", ["conv", "norm", "scan", "pscan"])       # (its node starts the second forward pass)
def test_operators_within_a_checkpoint(pkg, dev, last):
    """The forward pass that runs again inside the backward one is recorded like the first."""
    torch.manual_seed(2)
    Bs, L, ED, N = 2, 75, 96, 16
    rand = lambda *s: torch.randn(*s, device=dev).requires_grad_()
    x, z, raw, Bm, C, w, b, nw = (rand(Bs, L, ED), rand(Bs, L, ED), rand(Bs, L, ED), rand(Bs, L, N), rand(Bs, L, N), rand(ED, 4), rand(ED),
                                  rand(ED))
    A, D = torch.randn(ED, N, device=dev).requires_grad_(), rand(ED)
    leaves = [x, z, raw, Bm, C, w, b, nw, A, D]

    def f(x, z, raw, Bm, C, w, b, nw, A, D):
        u = pkg.causal_conv1d_fn(F.gelu(x), w.sin(), b.cos())
        if last == "conv":
            return u
        u = pkg.rmsnorm_fn(torch.tanh(u), nw.exp())
        if last == "norm":
            return u
        y = pkg.selective_scan_fn(torch.sin(u), F.softplus(raw), A.exp().neg(), Bm * 2, C * 2, D * 2, z=z.tanh())
        if last == "scan":
            return y
        wide = lambda t: t.unsqueeze(-1).expand(-1, -1, -1, 2)
        return pkg.pscan(wide(torch.sigmoid(y)), wide(y.cos()))

    y = f(*leaves)
    dy = torch.randn_like(y)
    want = torch.autograd.grad(y, leaves, dy, allow_unused=True)
    same = lambda got: all((a is None and b is None) or torch.equal(a, b) for a, b in zip(got, want))
    assert same(torch.autograd.grad(checkpoint(f, *leaves, use_reentrant=False), leaves, dy, allow_unused=True))
    with torch.autograd.graph.save_on_cpu():
        y = f(*leaves)
    assert same(torch.autograd.grad(y, leaves, dy, allow_unused=True))


def test_a_hook_that_changes_a_saved_tensor_is_refused(pkg, dev):
    blk = pkg.MambaBlock(pkg.MambaConfig(d_model=64, n_layers=1)).to(dev)
    x = torch.randn(2, 70, 64, device=dev, requires_grad=True)
    for change in (lambda t: t.to(torch.float64), lambda t: t[:1]):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, change):
            y = blk(x)
        with pytest.raises(RuntimeError, match="saved tensor"):
            y.sum().backward()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.unsqueeze(-1).expand(*t.shape, 2)[..., 0]):
        y = blk(x)          # the same values with other strides
    got = torch.autograd.grad(y.sum(), x)[0]
    assert torch.equal(got, torch.autograd.grad(blk(x).sum(), x)[0])
