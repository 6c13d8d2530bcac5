"""The float32 decode's split over workgroups (a merge adds the partials) against its one
workgroup per (kv head, sequence) and against float64, at the shapes where the stream's borders
matter: sequences shorter than a taker, longer than many, exactly a taker's share, none at all,
more than 64 sequences, a clamped table row, invalid blocks; lengths on both sides of the lines
where the workgroups take whole sequences (all short in a wide table, more of them than
workgroups; even ones that fill the GPU); batches appended by a launch of their own; with the
append, with RoPE and without either.

Split and whole sum the same fp32 terms in another order: a weighted mean of values of size
<= max|v| whose weights' relative error is at most (tiles + 8) 2^-24, so outputs differ by less
than 2 (tiles + 8) 2^-24 max|v|; the pool's bytes are the same.  Against float64 the scores' own
error comes on top (head_dim 2^-24 |q||k| scale, here < 64 2^-24): 2 (tiles + 80) 2^-24 max|v|.
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
    # whole sequences taken: the longest of 28 tiles (head_dim 64) or 18 (128), in a wide table
    "short-64": (14, 2, 64, 16, [447, 0, -1, 100, 5, 446], 90),
    "short-128": (28, 4, 128, 32, [3, 287, -2, 100, 286], 90),
    "short-many": (8, 4, 64, 16, [(53 * i) % 448 for i in range(150)], 60),
    "even": (32, 8, 128, 16, [640 + i % 9 for i in range(29)], 30),
    # one tile more than short, and one sequence too long for even
    "past-short-64": (14, 2, 64, 16, [448, 0, 100], 90),
    "past-short-128": (28, 4, 128, 16, [288, 17, 100, -1], 90),
    "past-even": (32, 8, 128, 16, [640 + i % 9 for i in range(28)] + [1500], 30),
}
# never split: rows appended by a launch before (768 workgroups, 64 sequences); tables of up to
# 40 and 64 tiles where the pairs fill the GPU once or twice
ONE_LAUNCH = {"full-once": (28, 4, 128, 16, [639 - 9 * i for i in range(50)], 0),
              "full-once-64": (14, 2, 64, 32, [1023 - 11 * i for i in range(64)], 0),
              "full-twice": (32, 32, 128, 16, [1023 - 31 * i for i in range(16)], 0),
              "append-first": (32, 8, 128, 16, [(7 * i) % 330 for i in range(95)] + [-1], 0),
              "append-first-64": (24, 12, 64, 16, [(11 * i) % 330 for i in range(64)], 0)}


def _inputs(case, form):
    h, hkv, d, bs, ctx, extra = case
    g = torch.Generator(device=DEV).manual_seed(7)
    n = len(ctx)
    blocks = [max(1, -(-(c + 1) // bs)) for c in ctx]
    width = max(blocks) + extra // (bs // 16 if extra < 0 else 1)
    if case in CASES.values():
        width = max(width, 52 * 16 // bs)   # past the single-workgroup sizes
    nb = n * width + 1
    pool = torch.randn(2, nb, hkv, bs, d, generator=g, device=DEV)
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(3))[:n * width]
    table = table.to(torch.int32).view(n, width)
    if case is CASES["mixed"]:
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
    return q, pool, table, lens, more


@pytest.mark.parametrize("form", ["plain", "append", "rope"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_split_equals_whole(name, form):
    h, hkv, d, bs, ctx, extra = CASES[name]
    q, pool, table, lens, more = _inputs(CASES[name], form)
    n, width = table.shape

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


def _rotate(x, cos, sin):   # float32, each product and the sum rounded
    half = x.shape[-1] // 2
    return x * cos[:, None] + torch.cat([-x[..., half:], x[..., :half]], -1) * sin[:, None]


@pytest.mark.parametrize("form", ["plain", "append", "rope"])
@pytest.mark.parametrize("name", sorted(CASES) + sorted(ONE_LAUNCH))
def test_vs_float64(name, form):
    case = CASES.get(name) or ONE_LAUNCH[name]
    h, hkv, d, bs, ctx, _ = case
    q, pool, table, lens, more = _inputs(case, form)
    n, width = table.shape
    nb = pool.shape[1]
    need = ops.decode_workspace_bytes(n, h, hkv, d, width, bs, 0, torch.float32)
    assert (need > 256) == (name in CASES)
    got_pool = pool.clone()
    got = ops.paged_decode(q, got_pool, table, lens, d ** -0.5, h, hkv, d, **more)
    want_pool, k, qr = pool.clone(), more.get("new_k"), q
    if form == "rope":
        qr, k = (_rotate(x, more["cos"], more["sin"]) for x in (q, k))
    rows = table.tolist()
    for i, c in enumerate(ctx):
        b = rows[i][min(c // bs, width - 1)] if c >= 0 else -1
        if form != "plain" and 0 <= b < nb:
            want_pool[0, b, :, c % bs], want_pool[1, b, :, c % bs] = k[i], more["new_v"][i]
    assert torch.equal(got_pool.view(torch.int32), want_pool.view(torch.int32))
    for i, c in enumerate(ctx):
        keys = min(c + 1, width * bs)
        if keys <= 0:
            assert not got[i].any()
            continue
        pos = torch.arange(keys, device=DEV)
        blk = table[i, pos // bs].long()
        ok = (blk >= 0) & (blk < nb)
        kv = want_pool[:, blk[ok], :, (pos % bs)[ok]].double()   # [keys, 2, hkv, d]
        ks, vs = kv.permute(1, 2, 0, 3).contiguous()
        w = torch.matmul(qr[i].double().view(hkv, h // hkv, d), ks.transpose(1, 2).contiguous())
        want = torch.matmul(torch.softmax(w * d ** -0.5, -1), vs).view(h, d)
        tol = 2 * (keys / 16 + 80) * 2.0 ** -24 * vs.abs().max().item()
        err = (got[i].double() - want).abs().max().item()
        assert err <= tol, (i, c, err, tol)
