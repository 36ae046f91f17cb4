"""The one-node mixer (csrc/host_train.cpp) and its weight-gradient kernel (csrc/layer.hip)."""
import ctypes

import pytest
import torch

from test_modules_gpu import block_forward_ref
from util import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("T", [1, 63, 65, 1000, 4097])                 # step edges; one and several parts of T
def test_weight_gradients_match_float64_products(pkg, dev, dtype, tol, T):
    L = pkg._lib
    g = torch.Generator().manual_seed(T)
    # (columns of P, of Q, kept columns, first row of the gap, gap): tile edges, both tile orders, padding
    sizes = [(8, 8, 8, 0, 0), (128, 136, 136, 0, 0), (264, 64, 17, 0, 0), (96, 392, 392, 17, 47)]
    jobs, keep, want, outs = (L.WgradJob * 4)(), [], [], []
    for j, (M, N, kept, at, gap) in zip(jobs, sizes):
        P = torch.randn(T, M + 16, generator=g).to(dtype).to(dev)[:, 8:8 + M]      # strided, offset
        Q = torch.randn(T, N, generator=g).to(dtype).to(dev)
        out = torch.full((M - gap, kept), float("nan"), dtype=dtype, device=dev)
        j.p, j.q, j.ldp, j.ldq, j.out = P.data_ptr(), Q.data_ptr(), P.stride(0), Q.stride(0), out.data_ptr()
        j.rows, j.cols, j.keep_cols, j.gap_at, j.gap = M, N, kept, at, gap
        ref = P.double().cpu().T @ Q.double().cpu()
        want.append(torch.cat([ref[:at], ref[at + gap:]])[:, :kept])
        keep += [P, Q]
        outs.append(out)
    lib, io = L.load(), pkg.scan._DTYPES[dtype]
    n = lib.mpa_wgrad_workspace_bytes(jobs, 4, T, io)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    L.check(lib.mpa_wgrad(jobs, 4, T, io, ctypes.c_void_p(ws.data_ptr()), n, pkg.scan._stream(dev)), "mpa_wgrad")
    for got, ref in zip(outs, want):
        assert rel_err(got, ref) <= tol
    jobs[0].rows = 10
    assert lib.mpa_wgrad(jobs, 4, T, io, ctypes.c_void_p(ws.data_ptr()), n, pkg.scan._stream(dev)) == 2


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-4), (torch.bfloat16, 5e-2)])
@pytest.mark.parametrize("shape,width,kw", [
    ((1, 3), 8, {}), ((2, 75), 48, {}), ((3, 130), 64, dict(d_state=8, d_conv=2)),
    ((2, 40), 72, dict(dt_rank=64, bias=False)), ((1, 33), 40, dict(d_state=32, d_conv=3, expand_factor=1)),
])
def test_mixer_gradients_match_float64_layer(pkg, dev, dtype, tol, shape, width, kw):
    torch.manual_seed(width)
    blk = pkg.MambaBlock(pkg.MambaConfig(d_model=width, n_layers=1, **kw)).to(dev).to(dtype)
    x = torch.randn(*shape, width).to(dtype)
    g = torch.randn(*shape, width).to(dtype)
    xr = x.double().requires_grad_()
    yr, pr = block_forward_ref(blk, xr)
    yr.backward(g.double())
    xg = x.to(dev).requires_grad_()
    y = blk(xg)
    assert "MambaBlockBackward" in type(y.grad_fn).__name__ or y.grad_fn.name() == "MambaBlockBackward"
    y.backward(g.to(dev), retain_graph=True)
    first = {k: v.grad.clone() for k, v in blk.named_parameters()}
    assert rel_err(y, yr) <= tol and rel_err(xg.grad, xr.grad) <= tol
    for k, v in blk.named_parameters():
        assert v.grad.dtype == v.dtype and rel_err(v.grad, pr[k].grad) <= 3 * tol, k
    # a second backward over the kept graph adds the same again; frozen parameters get none
    y.backward(g.to(dev))
    for k, v in blk.named_parameters():
        assert rel_err(v.grad, 2 * first[k].double()) <= 1e-2, k
    with pytest.raises(RuntimeError):
        y.backward(g.to(dev))
    for p in blk.parameters():
        p.grad = None
    blk.in_proj.weight.requires_grad_(False)
    blk(x.to(dev)).backward(g.to(dev))
    assert blk.in_proj.weight.grad is None
    assert all(rel_err(v.grad, first[k].double()) <= 1e-6 for k, v in blk.named_parameters() if v.grad is not None)
    # parameters changed between forward and backward are refused, as autograd does
    y = blk(x.to(dev))
    with torch.no_grad():
        blk.A_log.add_(1.0)
    with pytest.raises(RuntimeError):
        y.backward(g.to(dev))


# not whole 16-byte parts in either type; in bfloat16
@pytest.mark.parametrize("inner,dtype,tol", [(102, torch.float32, 2e-4), (102, torch.bfloat16, 5e-2), (100, torch.bfloat16, 5e-2)])
def test_mixer_of_any_inner_width(pkg, dev, inner, dtype, tol):
    torch.manual_seed(inner)
    cfg = pkg.MambaConfig(d_model=64, n_layers=1)
    cfg.d_inner = inner
    blk = pkg.MambaBlock(cfg).to(dev).to(dtype)
    x, g = torch.randn(2, 75, 64).to(dtype), torch.randn(2, 75, 64).to(dtype)
    xr = x.double().requires_grad_()
    yr, pr = block_forward_ref(blk, xr)
    yr.backward(g.double())
    xg = x.to(dev).requires_grad_()
    y = blk(xg)
    y.backward(g.to(dev))
    assert rel_err(y, yr) <= tol and rel_err(xg.grad, xr.grad) <= tol
    for k, v in blk.named_parameters():
        assert rel_err(v.grad, pr[k].grad) <= 3 * tol, k


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mixer_takes_operands_that_start_anywhere(pkg, dev, dtype):
    """Input and output gradient as views of flat buffers, one element off: the same results bit for bit."""
    torch.manual_seed(11)
    blk = pkg.MambaBlock(pkg.MambaConfig(d_model=64, n_layers=1)).to(dev).to(dtype)
    x, g = (torch.randn(2, 75, 64, device=dev).to(dtype) for _ in range(2))

    def off(t):
        v = torch.empty(t.numel() + 1, dtype=dtype, device=dev)[1:].view(t.shape)
        assert v.data_ptr() % 16
        return v.copy_(t)

    def run(x, g):
        x = x.detach().requires_grad_()
        y = blk(x)
        return [y.detach()] + list(torch.autograd.grad(y, [x] + list(blk.parameters()), g))
    want = run(x, g)
    for got in (run(off(x), g), run(x, off(g)), run(off(x), off(g))):
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_mixer_leaves_autocast_and_backward_hooks_to_the_composed_path(pkg, dev):
    torch.manual_seed(9)
    blk = pkg.MambaBlock(pkg.MambaConfig(d_model=64, n_layers=1)).to(dev)
    x = torch.randn(2, 50, 64, device=dev)
    y = blk(x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        ya = blk(x)
    assert ya.dtype == torch.bfloat16 and rel_err(ya, y.double()) <= 3e-2
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=1)).to(dev)(x).shape == x.shape
    seen = []
    blk.out_proj.register_full_backward_hook(lambda *_: seen.append(1))
    blk(x.requires_grad_()).sum().backward()
    assert seen == [1]
