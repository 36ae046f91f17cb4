"""Performance cases of the package: the calls its users make, over the sizes they make them at.

    listed()            the cases that are tracked by name
    draw(rng)           one more case from the same ranges
    prepare(case, seed) inputs, model and handle on the GPU, from the seed alone
    run(state)          one pass through the public entry points; returns everything it computes
    work(case)          bytes and operations that one pass cannot do without
    tolerance(case)     how far another correct implementation may be off

Kinds of case:
    scan     selective_scan_fn, forward and backward: the operator itself, as a training loop of
             one's own block calls it; plain, or with softplus(delta + bias) and the gate inside
    pscan    PScan.apply on materialised operands, forward and backward
    train    a stack of layers (Mamba), forward and backward: every parameter's gradient
    forward  LM over a batch of sequences without gradients: scoring, evaluation
    prefill  LM.prefill: a prompt in, the logits of its last position and the decode caches out
    decode   GraphedDecoder: one token per sequence through the whole model, step recorded once
    step     Mamba.step: one token per sequence, eager, caches returned as new tensors
"""
import math

import torch
import torch.nn.functional as F

import __graft_entry__

pkg = __graft_entry__.load_package()

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
VOCAB = 50280


def listed():
    return [
        # a layer of a toy model or a unit test: all launches and host work (B=2, L=64, 32 channels)
        dict(name="scan_tiny_f32", kind="scan", batch=2, length=64, channels=32, states=16, dtype="f32", gated=False),
        # one training layer in float32 (B=8, L=2048, 1536 channels)
        dict(name="scan_layer_f32", kind="scan", batch=8, length=2048, channels=1536, states=16, dtype="f32", gated=False),
        # the largest training layer, as a block calls it: bfloat16, softplus, bias and gate inside
        dict(name="scan_large_gated_bf16", kind="scan", batch=4, length=4096, channels=4096, states=16, dtype="bf16", gated=True),
        # batch 1, ragged length and width, wide state: few workgroups, several passes over the states
        dict(name="scan_thin_wide_f32", kind="scan", batch=1, length=3001, channels=1000, states=64, dtype="f32", gated=True),
        # the generic scan on (B, L, D, N) operands that do not fit any cache
        dict(name="pscan_large_f32", kind="pscan", batch=8, length=2048, channels=1536, states=16, dtype="f32"),
        # one block at batch 1 in float32, forward and backward: the regime of the README's plots
        dict(name="train_block_f32", kind="train", batch=1, length=4096, width=1024, layers=1, states=16, dtype="f32"),
        # training of a stack in bfloat16, a length that is no power of two
        dict(name="train_stack_bf16", kind="train", batch=8, length=1000, width=768, layers=4, states=16, dtype="bf16"),
        # scoring whole sequences with a 24-layer model, ragged length
        dict(name="forward_lm_bf16", kind="forward", batch=8, length=3000, width=768, layers=24, states=16, dtype="bf16"),
        # the prompt of one user: many small kernels
        dict(name="prefill_lm_b1_bf16", kind="prefill", batch=1, length=512, width=768, layers=24, states=16, dtype="bf16"),
        # serving: one token for one sequence, and for a batch
        dict(name="decode_lm_b1_bf16", kind="decode", batch=1, width=768, layers=24, states=16, dtype="bf16"),
        dict(name="decode_lm_b64_bf16", kind="decode", batch=64, width=768, layers=24, states=16, dtype="bf16"),
        # the eager step of a wide layer in float32, batch 64
        dict(name="step_layer_b64_f32", kind="step", batch=64, width=2560, layers=1, states=16, dtype="f32"),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], spread over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "pscan", "train", "train", "forward", "prefill", "decode", "decode", "step"])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "scan":
        states = rng.choice([16, 16, 16, 8, 24, 32, 64])
        while True:
            c = dict(kind=kind, batch=_log(rng, 1, 16), length=_log(rng, 50, 8192), channels=_log(rng, 32, 4096),
                     states=states, dtype=dtype, gated=rng.random() < 0.5)
            if c["batch"] * c["length"] * c["channels"] * states <= 4 * 4096 * 4096 * 16:
                return c
    if kind == "pscan":
        while True:
            c = dict(kind=kind, batch=_log(rng, 1, 16), length=_log(rng, 100, 65536), channels=_log(rng, 16, 1536),
                     states=rng.choice([8, 16, 16, 32]), dtype=dtype)
            if c["batch"] * c["length"] * c["channels"] * c["states"] <= 8 * 2048 * 1536 * 16:
                return c
    if kind == "train":
        while True:
            c = dict(kind=kind, batch=_log(rng, 1, 8), length=_log(rng, 100, 4096), width=8 * _log(rng, 8, 128),
                     layers=rng.randint(1, 4), states=16, dtype=dtype)
            if c["batch"] * c["length"] * c["width"] * c["layers"] <= (4 << 20) * (1 if dtype == "f32" else 6):
                return c
    model = dict(width=8 * _log(rng, 32, 96), layers=rng.randint(6, 24), states=16, dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "forward":
        while True:
            c = dict(kind=kind, batch=_log(rng, 1, 8), length=_log(rng, 200, 4096), **model)
            if c["batch"] * c["length"] <= (24000 if c["dtype"] == "bf16" else 4000):
                return c
    if kind == "prefill":
        while True:
            c = dict(kind=kind, batch=_log(rng, 1, 8), length=_log(rng, 32, 2048), **model)
            if c["batch"] * c["length"] <= 4096:
                return c
    if kind == "decode":
        return dict(kind=kind, batch=_log(rng, 1, 128), **model)
    return dict(kind=kind, batch=_log(rng, 1, 128), width=8 * _log(rng, 32, 320), layers=rng.randint(1, 4), states=16, dtype=dtype)


def _model(case, cls, gen_seed):
    torch.manual_seed(gen_seed)
    cfg = pkg.MambaConfig(d_model=case["width"], n_layers=case["layers"], d_state=case["states"])
    with torch.device("cuda"):
        m = cls(cfg) if cls is pkg.Mamba else cls(cfg, VOCAB, pad_vocab_size_multiple=8)
    return m.to(DTYPES[case["dtype"]]).eval()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    kind, B, N = case["kind"], case["batch"], case["states"]

    def normal(*shape, dtype=dt):
        return torch.randn(*shape, generator=g, device="cuda").to(dtype)

    if kind == "scan":
        L, ED = case["length"], case["channels"]
        # the values a layer starts from: A = -(1..N), steps log-uniform in [1e-3, 0.1], N(0, 1) inputs
        step = torch.exp(torch.rand(ED, generator=g, device="cuda") * math.log(100.0) + math.log(1e-3))
        bias = step + torch.log(-torch.expm1(-step))
        raw = 0.02 * torch.randn(B, L, ED, generator=g, device="cuda")
        s = dict(x=normal(B, L, ED), A=-torch.arange(1, N + 1, dtype=torch.float32, device="cuda").repeat(ED, 1),
                 B=normal(B, L, N), C=normal(B, L, N), D=torch.ones(ED, device="cuda"))
        if case["gated"]:
            s.update(delta=raw.to(dt), z=normal(B, L, ED), delta_bias=bias)
        else:
            s["delta"] = F.softplus(raw + bias).to(dt)
        return dict(kind=kind, leaves={k: v.requires_grad_() for k, v in s.items()}, softplus=case["gated"], dy=normal(B, L, ED))
    if kind == "pscan":
        shape = (B, case["length"], case["channels"], N)
        A = torch.rand(*shape, generator=g, device="cuda").mul_(0.5).add_(0.5).to(dt).requires_grad_()
        return dict(kind=kind, A=A, X=normal(*shape).requires_grad_(), dH=normal(*shape))
    if kind == "train":
        m = _model(case, pkg.Mamba, seed)
        x = normal(B, case["length"], case["width"]).requires_grad_()
        return dict(kind=kind, model=m, x=x, dy=normal(B, case["length"], case["width"]))
    if kind == "step":
        m = _model(case, pkg.Mamba, seed)
        ED, K = m.config.d_inner, m.config.d_conv
        caches = [(normal(B, ED, N, dtype=torch.float32), normal(B, ED, K - 1)) for _ in m.layers]
        return dict(kind=kind, model=m, x=normal(B, case["width"]), caches=caches)
    m = _model(case, pkg.LM, seed)
    if kind == "decode":
        ED, K = m.config.d_inner, m.config.d_conv
        caches = [(normal(B, ED, N, dtype=torch.float32), normal(B, ED, K - 1)) for _ in m.mamba.layers]
        token = torch.randint(0, VOCAB, (B,), generator=g, device="cuda")
        return dict(kind=kind, decoder=pkg.GraphedDecoder(m, caches), token=token, model=m)
    return dict(kind=kind, model=m, tokens=torch.randint(0, VOCAB, (B, case["length"]), generator=g, device="cuda"))


def run(s):
    kind = s["kind"]
    if kind == "scan":
        leaves = s["leaves"]
        for t in leaves.values():
            t.grad = None
        y = pkg.selective_scan_fn(**leaves, delta_softplus=s["softplus"])
        y.backward(s["dy"])
        return dict({"d" + k: t.grad for k, t in leaves.items()}, y=y)
    if kind == "pscan":
        A, X = s["A"], s["X"]
        A.grad = X.grad = None
        H = pkg.pscan(A, X)
        H.backward(s["dH"])
        return dict(H=H, dA=A.grad, dX=X.grad)
    if kind == "train":
        m, x = s["model"], s["x"]
        x.grad = None
        m.zero_grad(set_to_none=True)
        y = m(x)
        y.backward(s["dy"])
        return dict({k: p.grad for k, p in m.named_parameters()}, y=y, dx=x.grad)
    if kind == "forward":
        with torch.no_grad():
            return s["model"](s["tokens"])
    if kind == "prefill":
        logits, caches = s["model"].prefill(s["tokens"])
        return dict(logits=logits, caches=caches)
    if kind == "decode":
        logits = s["decoder"](s["token"])
        return dict(logits=logits, caches=s["decoder"].caches)
    with torch.no_grad():
        y, caches = s["model"].step(s["x"], list(s["caches"]))
    return dict(y=y, caches=caches)


# float32 operations per (batch, step, channel, state): forward delta*A, exp2, a*h + u*B, C*h;
# backward the recurrence again, g = dy*C + a*g, and the products of the five gradients
SCAN_FWD, SCAN_BWD = 7, 24


def _layer_flops(width, states, tokens):
    ED, R = 2 * width, -(-width // 16)
    gemm = 2 * tokens * (width * 2 * ED + ED * (R + 2 * states) + R * ED + ED * width)
    return gemm, tokens * ED * (SCAN_FWD * states + 2 * 4 + 10)


def work(case):
    s = 4 if case["dtype"] == "f32" else 2
    kind, B, N = case["kind"], case["batch"], case["states"]
    if kind == "scan":
        L, ED = case["length"], case["channels"]
        big, small = B * L * ED, B * L * N
        fwd = s * (3 * big + 2 * small) + 4 * (ED * N + ED)
        bwd = s * (5 * big + 4 * small) + 4 * (2 * ED * N + 2 * ED)
        if case["gated"]:
            fwd, bwd = fwd + s * big + 4 * ED, bwd + 2 * s * big + 8 * ED
        return dict(bytes=fwd + bwd, flops=big * N * (SCAN_FWD + SCAN_BWD))
    if kind == "pscan":
        n = B * case["length"] * case["channels"] * N
        return dict(bytes=8 * n * s, flops=5 * n)
    W, layers = case["width"], case["layers"]
    ED, R = 2 * W, -(-W // 16)
    weights = layers * (W * 2 * ED + ED * 5 + ED * (R + 2 * N) + R * ED + ED + ED * N + ED + ED * W + W)
    if kind == "train":
        T = B * case["length"]
        gemm, scan = _layer_flops(W, N, T)
        # weights read, their gradients written; x, dy in and y, dx out
        return dict(bytes=s * (2 * weights + 4 * T * W), flops=layers * (3 * gemm + scan * (SCAN_FWD + SCAN_BWD) / SCAN_FWD))
    state = layers * B * ED * (4 * N + s * 3)
    if kind == "step":
        gemm, scan = _layer_flops(W, N, B)
        return dict(bytes=s * (weights + 2 * B * W) + 2 * state, flops=layers * (gemm + scan))
    head = VOCAB * W
    if kind == "decode":
        gemm, scan = _layer_flops(W, N, B)
        return dict(bytes=s * (weights + head + W + B * W + B * VOCAB) + 2 * state, flops=layers * (gemm + scan) + 2 * B * head)
    T = B * case["length"]
    gemm, scan = _layer_flops(W, N, T)
    out = B if kind == "prefill" else T
    return dict(bytes=s * (weights + head + W + min(T, VOCAB) * W + out * VOCAB) + 8 * T + (state if kind == "prefill" else 0),
                flops=layers * (gemm + scan) + 2 * out * head)


def tolerance(case):
    # float32: sums of thousands of terms in another order, exp and log units of 1-2 ulp
    # bfloat16: roundings of 2^-9 at every tensor between two kernels, through up to 24 layers
    deep = case.get("layers", 1) > 1
    if case["dtype"] == "f32":
        return {"rel": 2e-5 if deep else 1e-5, "max": 1e-3}
    return {"rel": 2e-2 if deep else 1e-2, "max": 0.5}
