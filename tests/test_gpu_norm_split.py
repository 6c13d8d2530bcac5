"""RMSNorm with one wave and with four waves per row: the same call on both sides of the rules
(256 rows, hidden 2,048) and at chunk counts that leave lanes and waves without work, in place
and not, against float64.

Bound: the sum of squares has a relative error under hidden 2^-24, the reciprocal root, the two
products and their two roundings a few ulps: four ulps of the output's format.
"""
import pytest
import torch

from needle_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -20}


@pytest.mark.parametrize("dtype", sorted(ULP, key=str))
@pytest.mark.parametrize("hidden", [8, 504, 896, 2048, 2056, 3584, 8192])
@pytest.mark.parametrize("rows", [1, 5, 256, 257, 1030])
def test_norm(rows, hidden, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g, device=DEV).to(dtype)
    res = torch.randn(rows, hidden, generator=g, device=DEV).to(dtype)
    w = torch.randn(hidden, generator=g, device=DEV).to(dtype)
    for r in (None, res):
        got = ops.rms_norm(x, w, 1e-6, r)
        h = x if r is None else x + r
        if r is not None:
            assert torch.equal(got[1], h)
            got = got[0]
        want = h.double() * torch.rsqrt(h.double().pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
        err = (got.double() - want).abs() / (want.abs() + 2.0 ** -14)
        assert err.max().item() <= 4 * ULP[dtype], err.max().item()
    # the residual sum into the residual's own memory
    stream = torch.cuda.current_stream().cuda_stream
    out, inplace = torch.empty_like(x), res.clone()
    code = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}[dtype]
    rc = _lib.load().ndl_rms_norm(out.data_ptr(), inplace.data_ptr(), x.data_ptr(), hidden,
                                  inplace.data_ptr(), w.data_ptr(), rows, hidden, 1e-6, code,
                                  stream)
    assert rc == 0
    assert torch.equal(inplace, x + res) and torch.equal(out, ops.rms_norm(x, w, 1e-6, res)[0])
