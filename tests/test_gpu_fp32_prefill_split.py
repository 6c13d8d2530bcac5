"""The float32 prefill's two splits of a workgroup's waves (keys of 16 rows over four waves,
keys of 32 rows over two pairs) against float64, with fewer tiles than waves, prompts that end
inside a workgroup's rows, cached prefixes, uneven batches and an invalid block.

A row's output is a weighted mean of values of size <= max|v| whose weights' relative error is
at most (keys / 16 + 16) 2^-24 plus the scores' own (head_dim 2^-24 |q||k| scale, here < 64
2^-24): 2 (keys / 16 + 80) 2^-24 max|v|.
"""
import pytest
import torch

from needle_amd import ops
from test_gpu_prefill_split import _reference

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = {
    # name: (heads, kv heads, head_dim, page, [(cached, new)])
    "few": (14, 2, 64, 16, [(0, 1), (0, 15), (40, 17), (-2, 33)]),
    "prefix": (8, 2, 128, 32, [(700, 20), (0, 0), (64, 100)]),
    "many-even": (32, 8, 128, 16, [(0, 130), (16, 129), (0, 128), (5, 127), (0, 131), (0, 130),
                                   (0, 132)]),
    "many-64": (32, 32, 64, 64, [(0, 191), (30, 200), (0, 177), (0, 199), (100, 200)]),
    "uneven": (32, 8, 128, 16, [(0, 600), (0, 3), (0, 40), (9, 1)]),
}


def _check(name, rope, scale):
    h, hkv, d, bs, seqs = CASES[name]
    ctx, new = [c for c, _ in seqs], [n for _, n in seqs]
    g = torch.Generator(device=DEV).manual_seed(21)
    n_seq, total = len(seqs), sum(new)
    width = max(-(-(max(c, 0) + n) // bs) for c, n in seqs)
    nb = n_seq * width + 1
    pool = torch.randn(2, nb, hkv, bs, d, generator=g, device=DEV)
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(5))[:n_seq * width]
    table = table.to(torch.int32).view(n_seq, width)
    if name == "prefix":
        table[0, 3] = -1
    table = table.to(DEV)
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    cu = torch.tensor([0] + new, device=DEV).cumsum(0).to(torch.int32)
    q = torch.randn(total, h, d, generator=g, device=DEV)
    more, qr = {}, q
    if rope:
        ang = torch.rand(total, d // 2, generator=g, device=DEV) * 6.0
        ang = torch.cat([ang, ang], -1)
        more = dict(cos=ang.cos(), sin=ang.sin())
        rot = torch.cat([-q[..., d // 2:], q[..., :d // 2]], -1)
        qr = q * more["cos"][:, None] + rot * more["sin"][:, None]
    got = ops.varlen_prefill(q, pool, table, cu, lens, max(new), scale * d ** -0.5, h, hkv, d, **more)
    want = _reference(qr, pool, table, ctx, new, hkv, scale * d ** -0.5)
    keys = max(max(c, 0) + n for c, n in seqs)
    tol = 2 * (keys / 16 + 80) * 2.0 ** -24 * pool.abs().max().item()
    err = (got.double() - want).abs().max().item()
    assert err <= tol, (err, tol)


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_prefill_vs_fp64(name, rope):
    _check(name, rope, 1.0)


# A masked key stays masked whatever the sign of the scale (-inf times it is NaN or +inf), in
# both splits of the waves and beside an invalid block.
@pytest.mark.parametrize("scale", [0.0, -0.0, -1.0])
@pytest.mark.parametrize("name", ["few", "prefix", "many-even", "uneven"])
def test_scale_of_any_sign(name, scale):
    _check(name, False, scale)
