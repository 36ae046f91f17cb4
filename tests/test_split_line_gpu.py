"""Float32 layers around the line from which their wide products run on cut operands: values and every gradient against the parts of the
layer called one by one."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu


# 700 rows (half the harmonic mean) with 3 * 2^28 multiplications, 300 with 2^31; either side of each
@pytest.mark.parametrize("batch,length,width", [(1, 1391, 392), (2, 1337, 392), (3, 701, 516), (1, 1000, 600), (1, 8003, 380), (4, 2001, 200)])
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
