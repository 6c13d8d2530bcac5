"""The merge of a sequence's partials when eight waves share it, at the part counts where its
loops change (one part per wave, the prefetched eight, whole unrolled groups, more parts than
threads), against the per-sequence split, which has no partials, and the fp64 closed form.
"""
import pytest
import torch

from oracle import closed_form
from needle_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("heads,hkv,d", [(4, 1, 128), (3, 1, 64)])
@pytest.mark.parametrize("tiles", [2, 9, 16, 17, 64, 65, 129, 513, 1100])
def test_many_partials_of_one_sequence(tiles, heads, hkv, d):
    g = torch.Generator(device=DEV).manual_seed(tiles)
    n = 16 * tiles - 5
    pool = torch.randn(2, tiles + 1, hkv, 16, d, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(1, heads, d, generator=g, device=DEV).to(torch.bfloat16)
    # a width of at least 40 columns keeps 16 or more takers for the one sequence
    table = torch.zeros(1, max(tiles, 40), dtype=torch.int32, device=DEV)
    table[0, :tiles] = torch.randperm(tiles, generator=torch.Generator().manual_seed(1)).to(DEV)
    ctx = torch.tensor([n - 1], dtype=torch.int32, device=DEV)

    def run(part):
        return ops.paged_decode(q, pool, table, ctx, d ** -0.5, heads, hkv, d,
                                partition_tokens=part)
    got, whole = run(16), run(-1)   # one tile per partial / no partials
    want = torch.from_numpy(closed_form.decode_fp64(q.cpu(), pool.cpu(), table.cpu(), ctx.cpu(),
                                                    d ** -0.5, heads, hkv)).to(DEV)
    # Both paths round only P (2^-8 relative, averaged over n values) and the output
    # (2^-8): within three output half-ulps of each other and of fp64 at these magnitudes.
    for out in (got, whole):
        err = (out.double() - want).abs().max().item()
        assert err <= 3 * 2.0 ** -8 * want.abs().max().item() + 1e-4, err
