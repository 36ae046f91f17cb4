"""LM.forward without gradients: the head by the package's kernel where it takes it, by nn.Linear where anything wants to see the call."""
import pytest
import torch
import torch.nn as nn
from torch.utils.flop_counter import FlopCounterMode

from util import TOL, rel_err

pytestmark = pytest.mark.gpu


def _lm(pkg, dev, width=72, vocab=1000, dtype=torch.bfloat16):
    torch.manual_seed(width)
    return pkg.LM(pkg.MambaConfig(d_model=width, n_layers=1), vocab, pad_vocab_size_multiple=8).to(dev).to(dtype).eval()


@pytest.mark.parametrize("batch,length", [(1, 1), (3, 21), (1, 64), (2, 150), (5, 401)])
def test_logits(pkg, dev, batch, length):
    m = _lm(pkg, dev)
    tokens = torch.randint(0, 1000, (batch, length), device=dev)
    with torch.no_grad():
        h = m.norm_f(m.mamba(m.embedding(tokens)))
        got = m(tokens)
        taken = pkg.modules._host().linear_rows(m.lm_head, h) is not None
    assert taken == (batch * length >= 64) and got.shape == (batch, length, 1000)
    want = h.double() @ m.lm_head.weight.double().t()
    assert rel_err(got, want) <= TOL[torch.bfloat16] / 4


@pytest.mark.parametrize("rows", [(1, 256), (1, 400), (3, 333)])
def test_a_float32_head_is_float32(pkg, dev, rows):
    """A weight that selects columns gives these columns: whatever sums zeros and one value, in whatever order, keeps it."""
    m = _lm(pkg, dev, 1024, 8004, torch.float32)
    with torch.no_grad():
        h = torch.randn(*rows, 1024, device=dev)
        assert pkg.modules._host().linear_rows(m.lm_head, h) is None
        picked = torch.randint(0, 1024, (m.vocab_size,), device=dev)
        m.lm_head.weight.zero_()
        m.lm_head.weight[torch.arange(m.vocab_size, device=dev), picked] = 1.0
        tokens = torch.randint(0, 8004, rows, device=dev)
        h = m.norm_f(m.mamba(m.embedding(tokens)))
        assert torch.equal(m(tokens), h[..., picked])


def test_what_it_leaves_to_the_module(pkg, dev):
    m = _lm(pkg, dev)
    host, x = pkg.modules._host(), torch.randn(2, 100, 72, device=dev).bfloat16()
    head = m.lm_head
    with torch.no_grad():
        assert host.linear_rows(head, x) is not None
        assert host.linear_rows(head, x.float()) is None and host.linear_rows(head, x[..., :64]) is None
        assert host.linear_rows(head, x.transpose(0, 1)) is None and host.linear_rows(nn.Linear(72, 64).to(dev).bfloat16(), x) is None
        assert host.linear_rows(_lm(pkg, dev, dtype=torch.float32).lm_head, x) is None
        seen = []
        hook = head.register_forward_hook(lambda *a: seen.append(1))
        assert host.linear_rows(head, x) is None
        m(torch.zeros(2, 100, dtype=torch.long, device=dev))
        assert seen == [1]
        hook.remove()
        assert host.linear_rows(head, x) is not None
        head.forward = lambda v: v
        assert host.linear_rows(head, x) is None
        del head.forward
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert host.linear_rows(head, x) is None

        with FlopCounterMode(display=False) as counted:
            assert host.linear_rows(head, x) is None
            m.lm_head(x)
        assert counted.get_total_flops() == 2 * 200 * 72 * 1000

        class Other(nn.Linear):
            pass
        assert host.linear_rows(Other(72, 64, bias=False).to(dev).bfloat16(), x) is None
        with torch.inference_mode():
            assert host.linear_rows(head, x) is not None
    assert host.linear_rows(head, x) is None                       # gradients enabled
    m(torch.zeros(2, 100, dtype=torch.long, device=dev)).float().sum().backward()
    assert head.weight.grad is not None


def test_weight_changes_and_streams(pkg, dev):
    m = _lm(pkg, dev)
    tokens = torch.randint(0, 1000, (2, 100), device=dev)
    with torch.no_grad():
        a = m(tokens)
        m.lm_head.weight.mul_(2)
        b = m(tokens)
        m.lm_head.weight = nn.Parameter(m.lm_head.weight * 2)
        c = m(tokens)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            e = m(tokens)
        side.synchronize()
    assert torch.equal(b, 2 * a) and torch.equal(c, 4 * a) and torch.equal(e, c)
