"""The decode kernels (csrc/decode.hip) where their launches change: the pieces of a row that four, eight or sixteen waves take at
once and one more, a dt_rank that leaves x_proj's outputs no multiple of four, more than 64 of them, more partial sums than
a workgroup requests together, and the number of channels a lane owns."""
import pytest
import torch

from test_decode_gpu import layer_step_ref
from util import TOL, rel_err

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("dtype,batch,width,kw", [
    # in_proj of 12, 13, 24, 25 pieces; out_proj of 24, 26 and (expand_factor 1) as many as in_proj
    (BF16, 1, 768, {}), (BF16, 1, 776, {}), (BF16, 2, 1536, {}), (BF16, 2, 1544, {}),
    (F32, 1, 384, {}), (F32, 1, 388, {}), (F32, 3, 768, {}), (F32, 3, 772, {}),
    (BF16, 1, 768, dict(expand_factor=1)), (F32, 20, 384, dict(expand_factor=1)), (F32, 20, 392, dict(expand_factor=1)),
    # out_proj of 48 pieces and one more
    (BF16, 1, 1536, dict(dt_rank=8)), (BF16, 1, 1568, dict(dt_rank=8)), (F32, 17, 768, {}), (F32, 17, 784, {}),
    # dt_rank odd, below 16, above 64; 256 and more outputs of x_proj
    (BF16, 2, 256, dict(dt_rank=1)), (F32, 2, 256, dict(dt_rank=7)), (BF16, 5, 256, dict(dt_rank=65)), (F32, 2, 160, dict(dt_rank=130)),
    (BF16, 1, 128, dict(dt_rank=224)), (BF16, 1, 128, dict(dt_rank=225)), (F32, 16, 64, dict(dt_rank=480)),
    # one channel and four channels a lane; 192 channels, 12 partial sums; taps
    (F32, 8, 512, {}), (F32, 9, 512, {}), (BF16, 16, 96, dict(d_conv=3)), (F32, 4, 36, dict(d_conv=2, bias=True)),
])
def test_step_matches_float64_at_the_edges(pkg, dev, dtype, batch, width, kw):
    torch.manual_seed(width + batch)
    cfg = pkg.MambaConfig(d_model=width, n_layers=2, **kw)
    model = pkg.Mamba(cfg).to(dev).to(dtype)
    x = torch.randn(batch, width).to(dtype)
    caches = [(torch.randn(batch, cfg.d_inner, cfg.d_state), torch.randn(batch, cfg.d_inner, cfg.d_conv - 1).to(dtype))
              for _ in model.layers]
    xr, want = x.double(), []
    for layer, (h, w) in zip(model.layers, caches):
        y, h, w = layer_step_ref(layer, xr, h.double(), w.double())
        xr = xr + y
        want.append((h, w))
    with torch.no_grad():
        y, new = model.step(x.to(dev), [(h.to(dev), w.to(dev)) for h, w in caches])
    assert rel_err(y, xr) <= TOL[dtype]
    for (h, w), (hr, wr) in zip(new, want):
        assert rel_err(h, hr) <= TOL[dtype] and rel_err(w, wr) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_an_infinite_sequence_stays_alone(pkg, dev, dtype):
    """24 channels of d_model: the last row tile of out_proj is half empty, and its empty rows meet every sequence."""
    torch.manual_seed(5)
    model = pkg.Mamba(pkg.MambaConfig(d_model=24, n_layers=2)).to(dev).to(dtype)
    x = torch.randn(5, 24, device=dev).to(dtype)
    caches = [(torch.zeros(5, 48, 16, device=dev), torch.zeros(5, 48, 3, device=dev, dtype=dtype)) for _ in model.layers]
    with torch.no_grad():
        y0, c0 = model.step(x, list(caches))
        x[2] = float("inf")
        y1, c1 = model.step(x, list(caches))
    keep = [0, 1, 3, 4]
    assert torch.equal(y0[keep], y1[keep])
    for (h0, w0), (h1, w1) in zip(c0, c1):
        assert torch.equal(h0[keep], h1[keep]) and torch.equal(w0[keep], w1[keep])
    assert not torch.isfinite(y1[2].float()).any()


@pytest.mark.parametrize("width", [328, 376, 488])
def test_the_mean_of_squares_is_a_quotient(pkg, dev, width):
    """Rows of one value, whose squares and their sum are exact: their mean does not depend on the width, and neither does what in_proj, a selection
    of columns, leaves in the convolution's window.  (A product with a rounded 1 / width does.)"""
    def newest(d):
        m = pkg.Mamba(pkg.MambaConfig(d_model=d, n_layers=1, rms_norm_eps=1e-30)).to(dev)
        x = (torch.arange(9, 41, device=dev).float() / 16)[:, None].repeat(1, d)
        with torch.no_grad():
            w = m.layers[0].mixer.in_proj.weight
            w.zero_()
            w[torch.arange(w.size(0)), torch.arange(w.size(0)) % d] = 1.0
            return m.step(x, m.empty_caches(32, device=dev))[1][0][1][:, 0, -1]
    assert torch.equal(newest(width), newest(256))
