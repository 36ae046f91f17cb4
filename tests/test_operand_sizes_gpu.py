"""Operands whose size does not fit the others are refused before a launch: the kernels address every operand by the sizes of
x and A alone, and would read past the end of a shorter one."""
import pytest
import torch

pytestmark = pytest.mark.gpu

B, L, ED, N, K = 2, 6, 32, 16, 4


def t(*shape):
    g = torch.Generator().manual_seed(sum(shape) + len(shape))
    return (0.5 * torch.randn(*shape, generator=g)).cuda()


def scan_args(**kw):
    return {**dict(x=t(B, L, ED), delta=t(B, L, ED).abs(), A=-t(ED, N).abs(), B=t(B, L, N), C=t(B, L, N), D=t(ED), delta_softplus=True), **kw}


def step_args(**kw):
    return {**dict(x=t(B, ED), delta=t(B, ED).abs(), A=-t(ED, N).abs(), B=t(B, N), C=t(B, N), D=t(ED), delta_softplus=True), **kw}


def conv_args(**kw):
    return {**dict(x=t(B, L, ED), weight=t(ED, 1, K)), **kw}


def update_args(**kw):
    return {**dict(x=t(B, ED), window=t(B, ED, K - 1), weight=t(ED, 1, K)), **kw}


def norm_args(**kw):
    return {**dict(x=t(B, L, ED), weight=t(ED)), **kw}


WRONG = [
    ("selective_scan_fn", scan_args, "delta_bias", (1,)), ("selective_scan_fn", scan_args, "delta_bias", (ED - 1,)),
    ("selective_scan_fn", scan_args, "h0", (1, ED, N)), ("selective_scan_fn", scan_args, "h0", (B, ED, N - 1)),
    ("ssm_step", step_args, "delta", (1, ED)), ("ssm_step", step_args, "A", (ED - 1, N)), ("ssm_step", step_args, "B", (1, N)),
    ("ssm_step", step_args, "C", (B, N - 1)), ("ssm_step", step_args, "D", (1,)), ("ssm_step", step_args, "h", (1, ED, N)),
    ("ssm_step", step_args, "z", (1, ED)), ("ssm_step", step_args, "delta_bias", (1,)),
    ("causal_conv1d_fn", conv_args, "bias", (1,)), ("causal_conv1d_fn", conv_args, "bias", (ED - 1,)),
    ("causal_conv1d_update", update_args, "weight", (ED - 1, 1, K)), ("causal_conv1d_update", update_args, "bias", (1,)),
    ("causal_conv1d_update", update_args, "x", (B, 1, ED)),
    ("rmsnorm_fn", norm_args, "weight", (1,)), ("rmsnorm_fn", norm_args, "weight", (ED - 4,)), ("rmsnorm_fn", norm_args, "x", (B, 0)),
]


@pytest.mark.parametrize("fn,args,name,shape", WRONG, ids=[f"{f}-{n}{'x'.join(map(str, s))}" for f, _, n, s in WRONG])
def test_wrong_sizes_are_refused(pkg, fn, args, name, shape):
    fn = getattr(pkg, fn)
    fn(**args())                                     # (the same call in order)
    with pytest.raises(RuntimeError):
        fn(**args(**{name: torch.empty(shape, device="cuda")}))


def test_step_reads_rows_of_any_form(pkg):
    """B, C and z as (B, 1, n), (B, n, 1) and with a stride between the values of a row give what (B, n) gives: the same
    numbers in the same kernel, bit for bit."""
    z = t(B, ED)
    base = step_args()
    want = pkg.ssm_step(**base, z=z)
    for form in (lambda a: a.unsqueeze(1), lambda a: a.unsqueeze(2), lambda a: a.t().contiguous().t(),
                 lambda a: a.t().contiguous().t().unsqueeze(2)):
        got = pkg.ssm_step(**{**base, "B": form(base["B"]), "C": form(base["C"])}, z=form(z))
        assert all(torch.equal(g, w) for g, w in zip(got, want))
