"""The few-row linear kernel against the fp64 product, at the edges of its dispatch: rows per
16-row tile, the weight-tile counts where the split changes (256, 512 and 1024 tiles, and a
last workgroup whose tiles run past the columns), k shorter and longer than the ring.

Bound: operands are exact, products are summed in fp32 (k <= 8,256 terms in any order: error
<= k * 2^-24 * sum|x w|, and sum|x w| is about sqrt(k) times the result's standard deviation),
then one rounding (half an ulp: 2^-8 relative in bf16, whose significand has 8 bits, 2^-11 in
fp16).
"""
import pytest
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from needle_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _inputs(rows, n, k, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.05).to(dtype)
    b = torch.randn(n, generator=g, device=DEV).to(dtype)
    return x, w, b


def _check(got, want, mag, k, dtype):
    bound = EPS[dtype] * want.abs() + (k + 2) * 2.0 ** -24 * mag + 2.0 ** -24
    bad = (got.double() - want).abs() > bound
    assert not bad.any(), (int(bad.sum()), float(((got.double() - want).abs() / bound).max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 8, 15, 16, 17, 33, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(16, 64), (48, 320), (4096, 128), (4112, 192), (8192 + 16, 64),
                                 (16384 + 48, 64), (32, 8192 + 64)])
def test_linear(rows, n, k, dtype):
    x, w, b = _inputs(rows, n, k, dtype)
    assert ops.skinny_linear_takes(x, w, b)
    mag = x.double().abs() @ w.double().abs().t()
    want = x.double() @ w.double().t()
    _check(ops.linear(x, w), want, mag, k, dtype)
    _check(ops.linear(x, w, b), want + b.double(), mag + b.double().abs(), k, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 16, 17, 40, 64])
@pytest.mark.parametrize("inter,k", [(16, 64), (4096 + 16, 128), (4864, 896), (8192 + 48, 64)])
def test_linear_silu(rows, inter, k, dtype):
    x, w, _ = _inputs(rows, 2 * inter, k, dtype, 1)
    assert ops.skinny_linear_takes(x, w, None, 2)
    got = ops.linear_silu(x, w)
    gu = ops.linear(x, w)
    # the same sums (one split or another moves a rounding now and then), the same roundings
    want = ops.silu_mul(gu[:, :inter], gu[:, inter:])
    same = (got == want).double().mean().item()
    assert same > 0.98, same
    d = (got.double() - want.double()).abs()
    scale = gu[:, :inter].double().abs() * gu[:, inter:].double().abs()
    assert bool((d <= 8 * EPS[dtype] * (scale + want.double().abs()) + 1e-6).all())


def test_strided_rows_and_replays():
    x, w, b = _inputs(9, 1152, 896, torch.bfloat16, 2)
    wide = torch.full((9, 1024), float("nan"), device=DEV, dtype=torch.bfloat16)
    wide[:, 64:960] = x
    want = ops.linear(x, w, b)
    assert torch.equal(ops.linear(wide[:, 64:960], w, b), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.linear(x, w, b)
    for i in range(3):
        x.copy_(torch.randn_like(x))
        graph.replay()
        assert torch.equal(out, ops.linear(x, w, b)), i


def test_other_forms_keep_torchs_linear():
    x, w, b = _inputs(9, 64, 128, torch.bfloat16, 3)
    take = ops.skinny_linear_takes
    assert take(x, w, b)
    assert not take(x.float(), w.float(), b.float())
    assert not take(x[:0], w, b)
    assert not take(x.repeat(8, 1), w, b)                       # 72 rows
    assert not take(x[:, :96], w[:, :96].contiguous(), b)       # k not a multiple of 64
    assert not take(x[:, :64], w[:, :64], b)                    # strided weight
    assert not take(x, w[:40].contiguous(), b[:40].contiguous())
    assert not take(x.t().contiguous().t(), w, b)               # transposed rows
    assert not take(x.unsqueeze(0), w, b)
    wp = torch.nn.Parameter(w)
    assert not take(x, wp, b)
    with torch.no_grad():
        assert take(x, wp, b)
    with torch.autocast("cuda", dtype=torch.float16):
        assert not take(x, w, b)
    lin = F.linear(x.float(), wp.float(), b.float())
    y = ops.linear(x, wp, b)
    y.float().sum().backward()
    assert wp.grad is not None
    assert (y.float() - lin).norm() <= 1e-2 * lin.norm()


# Wide weights go to the library where the kernel's activations outweigh them; results stay
# F.linear's on both sides of the line.
@pytest.mark.parametrize("n,k,last", [(16384, 2048, 64), (16400, 2048, 32), (16400, 1024, 48),
                                      (16400, 512, 64)])
def test_rows_by_width(n, k, last):
    x, w, _ = _inputs(64, n, k, torch.bfloat16, 4)
    for rows in (32, last, min(last + 1, 64)):
        assert ops.skinny_linear_takes(x[:rows], w, None) == (rows <= last)
        assert ops.skinny_linear_takes(x[:rows], w[:16384], None, 2)
        mag = x[:rows].double().abs() @ w.double().abs().t()
        _check(ops.linear(x[:rows], w), x[:rows].double() @ w.double().t(), mag, k,
               torch.bfloat16)


class _Calls(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen = getattr(self, "seen", 0) + 1
        return func(*args, **(kwargs or {}))


class _Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen = getattr(self, "seen", 0) + (func is F.linear)
        return func(*args, **(kwargs or {}))


# What looks at the operation gets torch's own call, on tensors the kernel would take: a raw
# launch would lose the tangent, the traced node, the batch dimension, the mode's call.
@pytest.mark.parametrize("form", ["vmap", "dual", "trace", "dispatch", "function", "inference"])
def test_forms_of_a_call(form):
    x, w, b = _inputs(9, 64, 128, torch.bfloat16, 5)
    assert ops.skinny_linear_takes(x, w, b)
    takes, want = [], F.linear(x, w, b)

    def call(x):
        takes.append(ops.skinny_linear_takes(x, w, b))
        return ops.linear(x, w, b)
    if form == "vmap":
        xs = torch.stack([x, 2 * x])
        got, want = torch.func.vmap(call)(xs), torch.func.vmap(lambda x: F.linear(x, w, b))(xs)
    elif form == "dual":
        with forward_ad.dual_level():
            d = forward_ad.make_dual(x, torch.ones_like(x))
            got = forward_ad.unpack_dual(call(d)).tangent
            want = forward_ad.unpack_dual(F.linear(d, w, b)).tangent
    elif form == "trace":
        traced = torch.jit.trace(call, (x,), check_trace=False)
        y = torch.randn_like(x)
        got, want = traced(y), F.linear(y, w, b)
    elif form == "inference":     # not one of them: an ordinary call
        with torch.inference_mode():
            got = call(x)
        assert takes == [True]
        assert (got.float() - want.float()).norm() <= 1e-2 * want.float().norm()
        return
    else:
        with (_Calls() if form == "dispatch" else _Functions()) as mode:
            got = call(x)
        assert mode.seen >= 1
    assert takes and not any(takes)
    assert got.shape == want.shape and torch.equal(got, want)
    assert not ops.skinny_linear_takes(x, w.to_sparse_csr(), None)
