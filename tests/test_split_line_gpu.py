"""Float32 layers around the line from which their wide products run on cut operands: values and every gradient against the parts of the
layer called one by one; below it, products that keep every bit of a value."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu


# in_proj and out_proj on either side of 2.5 * 2^30 multiplications, and of 2^31 for the three of a backward
@pytest.mark.parametrize("batch,length,width", [(1, 1391, 392), (2, 1337, 392), (3, 701, 516), (1, 1000, 600), (1, 8003, 380), (4, 2001, 200), (1, 8003, 408), (1, 8003, 456),
                                                (3, 1401, 700)])
def test_layer(pkg, dev, batch, length, width, monkeypatch):
    torch.manual_seed(width)
    m = pkg.Mamba(pkg.MambaConfig(d_model=width, n_layers=1)).to(dev)
    x = torch.randn(batch, length, width, device=dev, requires_grad=True)
    dy = torch.randn(batch, length, width, device=dev)

    def run():
        x.grad = None
        m.zero_grad(set_to_none=True)
        y = m(x)
        y.backward(dy)
        with torch.no_grad():
            return dict({k: p.grad for k, p in m.named_parameters()}, y=y.detach(), dx=x.grad, plain=m(x))

    got = run()
    monkeypatch.setattr(pkg.modules, "PAD_PROJECTIONS", False)
    want = run()
    for k in want:
        # both sum up to 8003 float32 products: a rounding of 2^-24 a term at random is sqrt(8003) * 2^-24 = 5e-6 of the largest
        assert rel_err(got[k], want[k]) <= 2e-5, k


@pytest.mark.parametrize("batch,length,width", [(4, 2001, 200), (4, 850, 392), (2, 1001, 512)])
def test_products_below_the_line_keep_every_bit(pkg, dev, batch, length, width):
    """A mixer whose projections are selections, whose convolution is its newest tap and whose scan is D: nothing in it is a sum, so that what a batch
    row gives does not depend on the others, on the kernels or on the order of a sum, unless a product keeps less of a value than float32 does."""
    torch.manual_seed(width)
    m = pkg.MambaBlock(pkg.MambaConfig(d_model=width, n_layers=1)).to(dev)
    with torch.no_grad():
        for w in (m.in_proj.weight, m.out_proj.weight):
            w.zero_()
            w[torch.arange(w.size(0)), torch.arange(w.size(0)) % w.size(1)] = 1.0
        m.conv1d.weight.zero_()
        m.conv1d.weight[:, :, -1] = 1.0
        m.conv1d.bias.zero_()
        m.x_proj.weight.zero_()
    x, dy = torch.randn(batch, length, width, device=dev), torch.randn(batch, length, width, device=dev)

    def run(x, dy):
        x = x.clone().requires_grad_()
        y = m(x)
        y.backward(dy)
        return [y.detach(), x.grad]

    got, rows = run(x, dy), [run(x[i:i + 1], dy[i:i + 1]) for i in range(batch)]
    for k, v in enumerate(got):
        assert torch.equal(v, torch.cat([r[k] for r in rows]))
