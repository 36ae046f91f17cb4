"""Layers read their parameters as they are at the call: changed through .data (which leaves version counters
alone), under a captured graph, on another stream.  The yardstick is a deep copy made at the time of the call: it has
kept nothing from earlier ones, and runs the same kernels, so results are equal bit for bit."""
import copy

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


def train_pass(m, x, dy):
    y = m(x)
    return [y.detach()] + list(torch.autograd.grad(y, [x] + list(m.parameters()), dy))


def change(m, by=0.05):
    for i, p in enumerate(m.parameters()):
        p.data.add_(torch.full_like(p, by * (1 + i % 3)))


def same(a, b):
    return len(a) == len(b) and all(torch.equal(u, v) for u, v in zip(a, b))


# dt_rank: rounded up by zero rows and columns; a multiple of 64 as it is
@pytest.mark.parametrize("dt_rank", [5, 64])
@pytest.mark.parametrize("dtype", DTYPES)
def test_training_sees_writes_through_data(pkg, dev, dtype, dt_rank):
    torch.manual_seed(dt_rank)
    blk = pkg.MambaBlock(pkg.MambaConfig(d_model=64, n_layers=1, dt_rank=dt_rank)).to(dev).to(dtype)
    x = torch.randn(2, 70, 64, device=dev).to(dtype).requires_grad_()
    dy = torch.randn(2, 70, 64, device=dev).to(dtype)
    first = train_pass(blk, x, dy)
    versions = [p._version for p in blk.parameters()]
    for _ in range(2):
        change(blk)
        got, want = train_pass(blk, x, dy), train_pass(copy.deepcopy(blk), x, dy)
        assert same(got, want) and not torch.equal(got[0], first[0])
    assert versions == [p._version for p in blk.parameters()]


@pytest.mark.parametrize("dtype", DTYPES)
def test_calls_without_gradients_see_what_training_wrote(pkg, dev, dtype):
    torch.manual_seed(2)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev).to(dtype)
    x = torch.randn(2, 70, 64, device=dev).to(dtype)
    xr = x.clone().requires_grad_()

    @torch.no_grad()
    def frozen(m):
        y, caches = m.step(x[:, 0], m.empty_caches(2))
        y1, h, w = m.layers[0].mixer.step(x[:, 0], m.empty_caches(2)[0])[0], *caches[1]
        return [m(x), y, y1, h, w]

    first = frozen(m)
    for _ in range(2):
        train_pass(m, xr, torch.ones_like(x))
        change(m)
        got = frozen(m)
        assert same(got, frozen(copy.deepcopy(m))) and not torch.equal(got[0], first[0])


def test_captured_training_pass_sees_new_weights(pkg, dev):
    """Recorded once after warm-up passes, replayed after the weights have changed outside the graph."""
    torch.manual_seed(3)
    dtype = torch.bfloat16      # (no library products in either direction at this size)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev).to(dtype)
    x = torch.randn(2, 70, 64, device=dev).to(dtype).requires_grad_()
    dy = torch.randn(2, 70, 64, device=dev).to(dtype)
    side = torch.cuda.Stream(device=dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        for _ in range(3):
            train_pass(m, x, dy)
    torch.cuda.current_stream(dev).wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = train_pass(m, x, dy)
    for rep in range(3):
        with torch.no_grad():
            for i, p in enumerate(m.parameters()):
                p.add_(0.05 * (1 + (i + rep) % 3))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        assert same(got, train_pass(copy.deepcopy(m), x, dy)), rep
        torch.cuda.synchronize()


def test_training_on_two_streams(pkg, dev):
    """The second stream's call waits for nothing of the first one's, whose stream is busy."""
    torch.manual_seed(4)
    blk = pkg.MambaBlock(pkg.MambaConfig(d_model=64, n_layers=1)).to(dev).to(torch.bfloat16)
    x = torch.randn(2, 70, 64, device=dev).to(torch.bfloat16).requires_grad_()
    dy = torch.randn(2, 70, 64, device=dev).to(torch.bfloat16)
    want = train_pass(copy.deepcopy(blk), x, dy)
    busy = torch.randn(2048, 2048, device=dev)
    one, two = torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(one):
        for _ in range(40):
            busy = (busy @ busy).clamp_(-1, 1)
        a = train_pass(blk, x, dy)
    with torch.cuda.stream(two):
        b = train_pass(blk, x, dy)
    torch.cuda.synchronize()
    assert same(a, want) and same(b, want)


def test_inference_tensors_are_read_in_every_call(pkg, dev):
    """Parameters made under inference_mode have no version counter."""
    torch.manual_seed(5)
    with torch.inference_mode():
        m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev).to(torch.bfloat16)
        x = torch.randn(2, 30, 64, device=dev).to(torch.bfloat16)
        run = lambda m: [m(x), m.step(x[:, 0], m.empty_caches(2))[0]]
        first = run(m)
        for _ in range(2):
            for p in m.parameters():
                p.add_(0.05)
            got = run(m)
            assert same(got, run(copy.deepcopy(m))) and not torch.equal(got[0], first[0])


@torch.no_grad()
def forward_and_step(m, x):
    y, caches = m.step(x[:, 0], m.empty_caches(x.shape[0]))
    return [m(x), y] + [t for pair in caches for t in pair]


def test_a_stream_waits_for_the_forms_another_one_makes(pkg, dev):
    torch.manual_seed(6)
    m = pkg.Mamba(pkg.MambaConfig(d_model=64, n_layers=2)).to(dev).to(torch.bfloat16)
    x = torch.randn(2, 70, 64, device=dev).to(torch.bfloat16)
    want = forward_and_step(copy.deepcopy(m), x)
    one, two = torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)
    busy = torch.randn(2048, 2048, device=dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(one):
        for _ in range(40):
            busy = (busy @ busy).clamp_(-1, 1)
        a = forward_and_step(m, x)
    with torch.cuda.stream(two):
        b = forward_and_step(m, x)
    c = forward_and_step(m, x)
    torch.cuda.synchronize()
    assert same(a, want) and same(b, want) and same(c, want)


def test_a_capture_does_not_pass_for_a_run(pkg, dev):
    """Recorded on a model that has not run yet: the calls after it, before any replay, form the weights themselves."""
    torch.manual_seed(7)
    cfg = pkg.MambaConfig(d_model=64, n_layers=2)
    x = torch.randn(2, 70, 64, device=dev).to(torch.bfloat16)
    warm, m = (pkg.Mamba(cfg).to(dev).to(torch.bfloat16) for _ in range(2))
    forward_and_step(warm, x)
    want = forward_and_step(copy.deepcopy(m), x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = forward_and_step(m, x)
    assert same(forward_and_step(m, x), want)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, want)
        forward_and_step(warm, x)
        torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dt_rank", [16, 64])
def test_nothing_holds_the_parameters_between_calls(pkg, dev, dtype, dt_rank):
    """A model that moves to the host takes its memory along, but for the small forms; its tensors can be swapped."""
    torch.manual_seed(8)
    m = pkg.Mamba(pkg.MambaConfig(d_model=256, n_layers=3, dt_rank=dt_rank)).to(dev).to(dtype)
    x = torch.randn(2, 30, 256, device=dev).to(dtype)
    forward_and_step(m, x)
    train_pass(m, x.clone().requires_grad_(), torch.ones_like(x))
    forward_and_step(m, x)
    for layer in m.layers:
        for name in ("D", "A_log"):
            p = getattr(layer.mixer, name)
            torch.utils.swap_tensors(p, torch.nn.Parameter(p.detach() * 0.5))
        w = layer.mixer.in_proj.weight
        torch.utils.swap_tensors(w, torch.nn.Parameter(w.detach() * 2))
        torch.utils.swap_tensors(layer.norm.weight, torch.nn.Parameter(layer.norm.weight.detach() * 3))
    assert same(forward_and_step(m, x), forward_and_step(copy.deepcopy(m), x))
    for i in range(10):        # twice between two calls: the second new one may lie where the old one was
        for k in range(2):
            m.layers[0].mixer.A_log = torch.nn.Parameter(m.layers[0].mixer.A_log.detach() + 0.05 * (i + 3 * k))
            m.layers[0].norm.weight = torch.nn.Parameter(m.layers[0].norm.weight.detach() + 0.05 * (i + 3 * k))
        assert same(forward_and_step(m, x), forward_and_step(copy.deepcopy(m), x))
    torch.cuda.synchronize()
    weights = sum(p.numel() * p.element_size() for p in m.parameters())
    before = torch.cuda.memory_allocated(dev)
    m.to("cpu")
    assert before - torch.cuda.memory_allocated(dev) >= 0.95 * weights


def test_a_call_that_runs_out_of_memory(pkg, dev):
    """It fails with an exception, while forming the weights or after it; the next call, on another stream, is right."""
    torch.manual_seed(9)
    m = pkg.Mamba(pkg.MambaConfig(d_model=512, n_layers=4)).to(dev).to(torch.bfloat16)
    x = torch.randn(2, 4000, 512, device=dev).to(torch.bfloat16)
    want = forward_and_step(copy.deepcopy(m), x)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held, size = [], 256 << 20
    try:
        torch.cuda.set_per_process_memory_fraction(0.0, dev)
        while size >= 1 << 20:           # what is left free between the tensors of other tests
            try:
                held.append(torch.empty(size, dtype=torch.uint8, device=dev))
            except torch.cuda.OutOfMemoryError:
                size //= 2
        with pytest.raises(RuntimeError, match="out of memory"), torch.no_grad():
            m(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
        held.clear()
    stream = torch.cuda.Stream(device=dev)
    with torch.cuda.stream(stream):
        got = forward_and_step(m, x)
    torch.cuda.synchronize()
    assert same(got, want)
