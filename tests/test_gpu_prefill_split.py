"""The prefill whose tiles' keys are split over workgroups, against the launch of whole tiles
(ndl_varlen_prefill, no workspace) and float64, where the split's borders matter: pieces that
begin inside a 64-tile table window, tiles taken whole beside split ones, tiles whose causal
end lies in an earlier piece for some rows, sequences without tokens, partial last steps,
invalid blocks, a table row too short for the keys, larger pages.

Bound: P is rounded to 2^-9 of values up to 2^8 times its row's largest (averaged over the
keys), the output to half an ulp (2^-8 bf16, 2^-11 fp16): both launches are within 2 output
ulps of float64 at the scale of the values.
"""
import pytest
import torch

from needle_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = {
    # name: (heads, kv heads, head_dim, page, [(cached, new)], dtype, columns cut)
    "prefix": (32, 8, 128, 32, [(4001, 100), (900, 333), (2500, 64)], torch.bfloat16, 0),
    "one-prompt": (6, 1, 64, 16, [(0, 3000)], torch.float16, 0),
    "mixed": (28, 4, 128, 16, [(0, 5), (3000, 1), (0, 0), (777, 70), (-4, 33)], torch.bfloat16, 0),
    "mha": (8, 8, 64, 64, [(1023, 17), (2048, 31), (5000, 250)], torch.bfloat16, 0),
    "group-16": (16, 1, 128, 16, [(2234, 77), (0, 900)], torch.float16, 0),
    "short-table": (4, 2, 128, 16, [(1700, 90), (100, 200)], torch.bfloat16, 20),
}


def _reference(q, pool, table, ctx, new, hkv, scale):
    t, h, d = q.shape
    nb, bs = pool.shape[1], pool.shape[3]
    out = torch.zeros(t, h, d, dtype=torch.float64, device=DEV)
    at = 0
    for i, (c, n) in enumerate(zip(ctx, new)):
        if n == 0:
            continue
        c = max(c, 0)
        pos = torch.arange(c + n, device=DEV)
        tile = torch.clamp(pos // 16, max=table.shape[1] * bs // 16 - 1)   # the row's last tile
        row = tile * 16 + pos % 16
        blk = table[i, row // bs].long()
        ok = (blk >= 0) & (blk < nb)
        kv = pool[:, torch.where(ok, blk, 0), :, row % bs].double()   # [keys, 2, hkv, d]
        keys, vals = kv.permute(1, 2, 0, 3).contiguous()
        qi = q[at:at + n].double().view(n, hkv, h // hkv, d).permute(1, 2, 0, 3)
        w = torch.matmul(qi.reshape(hkv, -1, d), keys.transpose(1, 2).contiguous()) * scale
        w = w.view(hkv, h // hkv, n, c + n)
        mask = (pos > torch.arange(c, c + n, device=DEV)[:, None]) | ~ok
        w = torch.softmax(w.masked_fill(mask, float("-inf")), -1)
        o = torch.matmul(w.view(hkv, -1, c + n), vals).view(hkv, h // hkv, n, d)
        out[at:at + n] = o.permute(2, 0, 1, 3).reshape(n, h, d)
        at += n
    return out


def _check(name, rope, scale):
    h, hkv, d, bs, seqs, dtype, cut = CASES[name]
    scale *= d ** -0.5
    ctx, new = [c for c, _ in seqs], [n for _, n in seqs]
    g = torch.Generator(device=DEV).manual_seed(11)
    width = max(max(-(-(max(c, 0) + n) // bs) for c, n in seqs), 800 // bs) - cut
    n_seq, total = len(seqs), sum(new)
    nb = n_seq * width + 1
    pool = torch.randn(2, nb, hkv, bs, d, generator=g, device=DEV).to(dtype)
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(5))[:n_seq * width]
    table = table.to(torch.int32).view(n_seq, width)
    if name == "mixed":
        table[1, 40], table[3, 20] = -1, nb
    table = table.to(DEV)
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    cu = torch.tensor([0] + new, device=DEV).cumsum(0).to(torch.int32)
    q = torch.randn(total, h, d, generator=g, device=DEV).to(dtype)
    cos = sin = None
    if rope:
        ang = torch.rand(total, d // 2, generator=g, device=DEV) * 6.0
        ang = torch.cat([ang, ang], -1)
        cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    lib = _lib.load()
    code = {torch.bfloat16: 0, torch.float16: 1}[dtype]
    assert lib.ndl_varlen_prefill_workspace_bytes(n_seq, total, max(new), width, h, hkv, d, bs, code)
    got = ops.varlen_prefill(q, pool, table, cu, lens, max(new), scale, h, hkv, d,
                             max_context_len=max(max(ctx), 0), cos=cos, sin=sin)
    whole = torch.empty_like(got)
    rc = lib.ndl_varlen_prefill_split(
        whole.data_ptr(), q.data_ptr(), h * d, cos.data_ptr() if rope else None,
        sin.data_ptr() if rope else None, d, pool.data_ptr(), nb, table.data_ptr(), width, width,
        cu.data_ptr(), lens.data_ptr(), n_seq, total, max(new), max(max(ctx), 0), h, hkv, d, bs, code,
        scale, None, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    qr = q
    if rope:
        rot = torch.cat([-q[..., d // 2:], q[..., :d // 2]], -1)
        qr = q * cos[:, None] + rot * sin[:, None]
    want = _reference(qr, pool, table, ctx, new, hkv, scale)
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    for what, out in (("whole", whole), ("split", got)):
        assert torch.isfinite(out).all(), what
        err = (out.double() - want).abs() - 2 * ulp * want.abs()
        bad = (err > 2 * ulp).flatten(1).any(1).nonzero().flatten().tolist()
        assert not bad, (what, len(bad), bad[:8], err.max().item())


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_split_equals_whole_tiles(name, rope):
    _check(name, rope, 1.0)


# A masked key stays masked whatever the sign of the scale (-inf times it is NaN or +inf).
@pytest.mark.parametrize("scale", [0.0, -0.0, -1.0])
@pytest.mark.parametrize("name,rope", [("prefix", True), ("one-prompt", False), ("mixed", False),
                                       ("short-table", True)])
def test_scale_of_any_sign(name, rope, scale):
    _check(name, rope, scale)


# The choice counts the keys a sequence can have (max_context_len + max_seqlen), not the table's
# columns: a short prompt in a table of the model's length runs as in a tight one, without the
# pieces' workspace; with the bound of a long prefix the pieces are there.
@pytest.mark.parametrize("native", [True, False])
def test_wide_table_is_not_a_long_prompt(monkeypatch, native):
    _lib.load()
    if not native:
        monkeypatch.setattr(_lib, "NATIVE", None)
    h, hkv, d, bs, n, wide = 14, 2, 64, 16, 301, 256
    g = torch.Generator(device=DEV).manual_seed(3)
    pool = torch.randn(2, wide, hkv, bs, d, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(n, h, d, generator=g, device=DEV).to(torch.bfloat16)
    table = torch.randperm(wide, generator=torch.Generator().manual_seed(5)).to(torch.int32)
    table = table.view(1, wide).to(DEV)
    lens = torch.zeros(1, dtype=torch.int32, device=DEV)
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)

    def run(table, cached):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out = ops.varlen_prefill(q, pool, table, cu, lens, n, d ** -0.5, h, hkv, d,
                                 max_context_len=cached)
        return out, torch.cuda.max_memory_allocated() - before
    tight, _ = run(table[:, :19].contiguous(), 0)
    out, used = run(table, 0)
    assert torch.equal(out, tight) and used < 2 * out.numel() * 2
    _, used = run(table, 3700)
    assert used > 16 << 20
    with pytest.raises(_lib.NeedleAmdError):   # an empty block: the launch's own error
        ops.varlen_prefill(q, pool[:, :, :, :0], table, cu, lens, n, d ** -0.5, h, hkv, d)
