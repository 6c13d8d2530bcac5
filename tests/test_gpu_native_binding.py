"""The native bindings against ops.py's own path: the same bytes for the calls they take, and
None (so that ops.py's checks answer) for the others, over dtypes, strides and wrong arguments.
"""
import pytest
import torch

from needle_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


@pytest.fixture()
def native():
    _lib.load()
    assert _lib.NATIVE is not None
    return _lib.NATIVE


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _both(monkeypatch, call):
    """(result through the bindings, result of ops.py alone); an exception stands as its type."""
    def run():
        try:
            return call()
        except Exception as e:   # noqa: BLE001 - compared, not handled
            return type(e)
    fast = run()
    monkeypatch.setattr(_lib, "NATIVE", None)
    slow = run()
    monkeypatch.undo()
    return fast, slow


def _same(a, b):
    if isinstance(a, type) or isinstance(b, type) or a is None or b is None:
        assert a is b
    elif isinstance(a, tuple):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
        assert torch.equal(_bytes(a), _bytes(b))


@pytest.mark.parametrize("dtype", DTYPES)
def test_norm_and_silu(native, monkeypatch, dtype):
    g = torch.Generator(device=DEV).manual_seed(1)
    wide = torch.randn(9, 2 * 896, generator=g, device=DEV).to(dtype)
    x, w = wide[:, 896:], torch.randn(896, generator=g, device=DEV).to(dtype)
    res = torch.randn(9, 896, generator=g, device=DEV).to(dtype)
    assert native.rms_norm(x, w, 1e-6, res) is not None
    odd = {"shifted": wide[:, 1:897], "cpu": x.cpu(), "3d": x.unsqueeze(0), "no rows": x[:0],
           "transposed": torch.randn(896, 9, device=DEV).to(dtype).t(), "double": x.double()}
    for bad in odd.values():
        assert native.rms_norm(bad, w, 1e-6, None) is None
        _same(*_both(monkeypatch, lambda: ops.rms_norm(bad, w, 1e-6)))
    for r in (None, res, res[:8], res.t(), wide[:, :896], res.double()):
        _same(*_both(monkeypatch, lambda: ops.rms_norm(x, w, 1e-6, r)))
    for ww in (w[:888], w.double(), wide[0, ::2], w.cpu()):
        _same(*_both(monkeypatch, lambda: ops.rms_norm(x, ww, 1e-6)))
    _same(*_both(monkeypatch, lambda: ops.rms_norm(x, w, 1)))          # an int eps
    assert native.silu_mul(wide[:, :896], x) is not None
    for a, b in ((wide[:, :896], x), (x, x[:8]), (wide[:, 1:897], x), (x, x.double()),
                 (x[:1], wide[3:4, :896]), (x[:0], x[:0])):
        _same(*_both(monkeypatch, lambda: ops.silu_mul(a, b)))


@pytest.mark.parametrize("dtype", DTYPES)
def test_append_and_prefill(native, monkeypatch, dtype):
    g = torch.Generator(device=DEV).manual_seed(2)
    h, hkv, d, bs, new, ctx = 4, 2, 64, 16, [33, 0, 5], [7, 3, 900]
    n = sum(new)
    qkv = torch.randn(n, (h + 2 * hkv) * d, generator=g, device=DEV).to(dtype)
    q, k, v = qkv.split([h * d, hkv * d, hkv * d], dim=-1)
    q, k, v = q.view(n, h, d), k.view(n, hkv, d), v.view(n, hkv, d)
    pool0 = torch.randn(2, 200, hkv, bs, d, generator=g, device=DEV).to(dtype)
    table = torch.randperm(200, generator=torch.Generator().manual_seed(3))[:3 * 57]
    table = table.to(torch.int32).view(3, 57).to(DEV)
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    cu = torch.tensor([0] + new, device=DEV).cumsum(0).to(torch.int32)
    ang = torch.rand(n, d, generator=g, device=DEV)
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)

    def append(k=k, v=v, cos=cos, sin=sin, table=table, lens=lens, cu=cu):
        pool = pool0.clone()
        assert ops.rope_kv_append(None, k, v, cos, sin, pool, table, lens, cu) is None
        return pool

    def prefill(q=q, table=table, cu=cu, lens=lens, most=33, scale=0.125, cos=cos, sin=sin, h=h):
        return ops.varlen_prefill(q, pool0, table, cu, lens, most, scale, h, hkv, d,
                                  max_context_len=900, cos=cos, sin=sin)
    assert native.rope_kv_append(k, v, cos, sin, pool0.clone(), table, lens, cu)
    assert native.varlen_prefill(q, pool0, table, cu, lens, 33, 0.125, h, hkv, d, 900, cos,
                                 sin) is not None
    changes = [dict(), dict(cos=cos[:5]), dict(cos=cos.double()), dict(sin=sin.cpu()),
               dict(table=table.long()), dict(lens=lens[:2]), dict(cu=cu[:3]),
               dict(table=table[:, ::2]), dict(table=table[:, :0]), dict(cu=cu.long())]
    for change in changes + [dict(k=k[:5]), dict(v=v.transpose(0, 1)), dict(k=k.double())]:
        _same(*_both(monkeypatch, lambda: append(**change)))
    for change in changes + [dict(q=q[:5]), dict(q=q.double()), dict(cos=None, sin=None),
                             dict(cos=None), dict(scale=1), dict(most=0), dict(h=3),
                             dict(most=torch.tensor(33)), dict(q=q[..., :32])]:
        a, b = _both(monkeypatch, lambda: prefill(**change))
        if change.get("most") == 0 and not isinstance(change.get("most"), torch.Tensor):
            continue   # nothing is computed: the output's bytes are whatever was there
        _same(a, b)
