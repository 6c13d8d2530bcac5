"""The float32 decode's split over workgroups (a merge adds the partials) against its one
workgroup per (kv head, sequence), at the shapes where the stream's borders matter: sequences
shorter than a taker, longer than many, exactly a taker's share, none at all, more than 64
sequences, a clamped table row, invalid blocks; with the append, with RoPE and without either.

Both sum the same fp32 terms in another order: a weighted mean of values of size <= max|v|
whose weights' relative error is at most (tiles + 8) 2^-24, so outputs differ by less than
2 (tiles + 8) 2^-24 max|v|; the pool's bytes are the same.
"""
import pytest
import torch

from needle_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = {
    # name: (heads, kv heads, head_dim, block size, contexts, table columns beyond the longest)
    "mixed": (28, 4, 128, 16, [0, 15, 16, 100, 4000, -1, 271, 1023, 511, 2048], 0),
    "one-long": (8, 8, 64, 16, [9001], 3),
    "many-short": (14, 2, 64, 16, [(37 * i) % 700 for i in range(130)], 20),
    "page-64": (32, 8, 128, 64, [63, 64, 65, 3000, 700], 1),
    "group-16": (16, 1, 128, 32, [2000, 1, 900], 0),
    "clamped": (4, 2, 64, 32, [5000, 640, 2559, 2560, 3], -160),
}


@pytest.mark.parametrize("form", ["plain", "append", "rope"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_split_equals_whole(name, form):
    h, hkv, d, bs, ctx, extra = CASES[name]
    g = torch.Generator(device=DEV).manual_seed(7)
    n = len(ctx)
    blocks = [max(1, -(-(c + 1) // bs)) for c in ctx]
    width = max(blocks) + extra // (bs // 16 if extra < 0 else 1)
    width = max(width, 52 * 16 // bs)   # past the single-workgroup sizes
    nb = n * width + 1
    pool = torch.randn(2, nb, hkv, bs, d, generator=g, device=DEV)
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(3))[:n * width]
    table = table.to(torch.int32).view(n, width)
    if name == "mixed":
        table[4, 7], table[7, 0] = -3, nb + 5      # never read; their keys are dropped
    table = table.to(DEV)
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    q = torch.randn(n, h, d, generator=g, device=DEV)
    more = {}
    if form != "plain":
        more = dict(new_k=torch.randn(n, hkv, d, generator=g, device=DEV),
                    new_v=torch.randn(n, hkv, d, generator=g, device=DEV))
    if form == "rope":
        ang = torch.rand(n, d // 2, generator=g, device=DEV) * 6.0
        ang = torch.cat([ang, ang], -1)
        more.update(cos=ang.cos(), sin=ang.sin())

    def run(part):
        p = pool.clone()
        return ops.paged_decode(q, p, table, lens, d ** -0.5, h, hkv, d, partition_tokens=part,
                                **more), p
    assert ops.decode_workspace_bytes(n, h, hkv, d, width, bs, 0, torch.float32) > 256
    got, pool_got = run(0)
    want, pool_want = run(-1)
    assert torch.equal(pool_got.view(torch.int32), pool_want.view(torch.int32))
    tiles = -(-min(max(ctx) + 1, width * bs) // 16)
    tol = 2 * (tiles + 8) * 2.0 ** -24 * max(pool.abs().max().item(), 6.0)
    err = (got - want).abs().max().item()
    assert err <= tol, (err, tol)
    for i, c in enumerate(ctx):
        if c < 0:
            assert not got[i].any()
