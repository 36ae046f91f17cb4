"""Decode steps (csrc/decode.hip): float32 at rows that are not whole eights, and where in_proj's forms change."""
import pytest
import torch

import test_decode_gpu
from test_decode_gpu import layer_step_ref
from util import rel_err

pytestmark = pytest.mark.gpu


def both(pkg, dev, batch, width, kw):
    torch.manual_seed(batch * 1000 + width)
    cfg = pkg.MambaConfig(d_model=width, n_layers=2, **kw)
    model = pkg.Mamba(cfg).to(dev)
    x = torch.randn(batch, width, device=dev)
    with torch.no_grad():
        for layer in model.layers:
            layer.norm.weight.uniform_(0.5, 1.5)
    caches = [(torch.randn(batch, cfg.d_inner, cfg.d_state, device=dev), torch.randn(batch, cfg.d_inner, cfg.d_conv - 1, device=dev))
              for _ in model.layers]
    xr = x.double().cpu()
    want = []
    for layer, (h, w) in zip(model.layers, caches):
        y, h, w = layer_step_ref(layer, xr, h.double().cpu(), w.double().cpu())
        xr = xr + y
        want.append((h, w))
    with torch.no_grad():
        y, new = model.step(x, list(caches))
    return y, new, xr, want


# Rows of eight values and a half (d_model and d_inner not multiples of 8), of several pieces; every form of the kernels: one
# batch tile with x_proj inside, x_proj of its own, two tiles a workgroup, rows scaled by a launch of their own.  A float32 layer is
# a few roundings of 2^-24 on sums of up to 2056 terms, sqrt(2056) of them: below 1e-5 of the largest result.
@pytest.mark.parametrize("batch,width,kw", [(1, 4, {}), (1, 20, dict(expand_factor=1)), (5, 132, dict(expand_factor=1)), (17, 132, {}),
                                            (33, 1028, dict(expand_factor=1)), (65, 1028, {}), (128, 1028, dict(dt_rank=20))])
def test_float32_step_matches_float64(pkg, dev, batch, width, kw):
    y, new, yr, want = both(pkg, dev, batch, width, kw)
    assert rel_err(y, yr) <= 1e-5
    for (h, w), (hr, wr) in zip(new, want):
        assert rel_err(h, hr) <= 1e-5 and rel_err(w, wr) <= 1e-5


# The lines between in_proj's forms with x_proj inside: up to 256, 512 and 704 columns.
@pytest.mark.parametrize("batch,width", [(1, 256), (7, 260), (16, 512), (1, 516), (3, 700), (16, 704)])
def test_float32_step_at_the_lines_of_in_proj(pkg, dev, batch, width):
    test_float32_step_matches_float64(pkg, dev, batch, width, {})


# x_proj inside in_proj takes a thread for each of its dt_rank + 2 * d_state rows: more of them than four waves have, as many,
# and the most that are taken at this width.
@pytest.mark.parametrize("batch,width,kw", [(1, 704, dict(d_state=128)), (16, 704, dict(d_state=128)), (5, 768, dict(d_state=112, dt_rank=33)),
                                            (5, 768, dict(d_state=112, dt_rank=32)), (2, 704, dict(d_state=128, dt_rank=116))])
def test_float32_step_with_many_rows_of_x_proj(pkg, dev, batch, width, kw):
    test_float32_step_matches_float64(pkg, dev, batch, width, dict(kw, expand_factor=1))


# Few rows of x_proj over many channels: its partial sums, one per 16 channels, are 256 and 512, and the batch is large enough that
# the state kernel would take two and four sequences a workgroup.
@pytest.mark.parametrize("batch,width,kw", [(16, 512, dict(d_state=16, dt_rank=32)), (13, 1024, dict(d_state=8, dt_rank=8))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_step_of_many_channels_matches_float64(pkg, dev, dtype, batch, width, kw):
    test_decode_gpu.test_stack_step_matches_float64_layers(pkg, dev, dtype, batch, width, dict(kw, expand_factor=8))


# bfloat16, two batch tiles a workgroup: up to 1024 columns on four waves, then on eight.
@pytest.mark.parametrize("batch,width", [(97, 1024), (128, 1000), (97, 1032)])
def test_bfloat16_step_at_the_line_of_in_proj(pkg, dev, batch, width):
    test_decode_gpu.test_stack_step_matches_float64_layers(pkg, dev, torch.bfloat16, batch, width, {})
