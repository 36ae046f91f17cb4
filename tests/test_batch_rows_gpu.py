"""What one batch row holds does not reach the others: sequences that end inside a tile, next to one with NaN or infinity."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# lengths with a remainder (tiles of 16 steps); a short sequence whose tile spans several rows, one that is cut into segments (both
# passes, and the carry of the backward); states in one pass and in two, with and without a power of two; layers whose scan
# forms delta itself (bfloat16, up to 16 states)
@pytest.mark.parametrize("length,width,states", [(1, 64, 16), (3, 24, 4), (33, 72, 17), (130, 64, 16), (130, 32, 80), (1000, 64, 16), (1000, 32, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_rows_are_apart(pkg, dev, length, width, states, dtype, value):
    torch.manual_seed(length)
    m = pkg.Mamba(pkg.MambaConfig(d_model=width, n_layers=2, d_state=states)).to(dev).to(dtype)
    x = torch.randn(4, length, width, device=dev).to(dtype)
    g = torch.randn(4, length, width, device=dev).to(dtype)
    bad, bad_g = x.clone(), g.clone()
    bad[2], bad_g[1, length // 2:] = value, value
    rows = [0, 3]

    def run(x, g):
        with torch.no_grad():
            y, caches = m(x, return_caches=True)
        leaf = x.clone().requires_grad_()
        out = m(leaf)
        out.backward(g)
        return [y, out.detach(), leaf.grad, *(t for c in caches for t in c)]

    for a, b in zip(run(x, g), run(bad, bad_g)):
        assert a.isfinite().all() and torch.equal(a[rows], b[rows])
    for a, b in zip(run(x, g)[3:], run(bad, g)[3:]):  # (states and windows of the row in front as well)
        assert torch.equal(a[:2], b[:2])


# the operator on rows of a longer buffer: what lies behind a row's end is no part of it
@pytest.mark.parametrize("length", [5, 70, 1000])
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("gated", [False, True])
def test_views_of_a_longer_buffer(pkg, dev, length, reverse, gated):
    torch.manual_seed(length)
    B, ED, N, room = 3, 40, 16, length + 20
    def rows(*shape, scale=1.0):
        buf = torch.full((B, room, *shape), float("nan"), device=dev)
        buf[:, :length] = scale * torch.randn(B, length, *shape, device=dev)
        return buf
    bufs = dict(x=rows(ED), delta=rows(ED, scale=0.1).abs_(), B=rows(N), C=rows(N), z=rows(ED))
    A, D = -torch.arange(1.0, N + 1, device=dev).repeat(ED, 1), torch.ones(ED, device=dev)
    dy = rows(ED)

    def run(take):
        leaves = {k: take(v).requires_grad_() for k, v in bufs.items() if gated or k != "z"}
        y = pkg.selective_scan_fn(A=A, D=D, reverse=reverse, **leaves)
        return [y, *torch.autograd.grad(y, list(leaves.values()), take(dy))]

    for a, b in zip(run(lambda t: t[:, :length].detach()), run(lambda t: t[:, :length].contiguous())):
        assert b.isfinite().all() and torch.equal(a, b)
