"""A decode workspace sized without a dtype serves every dtype, as it did when all had one size."""
import pytest
import torch

from needle_amd import ops

SHAPES = [(2, 32, 8, 128, 64, 16), (12, 28, 4, 128, 251, 16), (1, 14, 2, 64, 2048, 16),
          (130, 14, 2, 64, 63, 16), (3, 32, 32, 128, 40, 64), (64, 8, 8, 64, 49, 16)]


@pytest.mark.parametrize("shape", SHAPES)
def test_default_size_covers_every_dtype(shape):
    both = ops.decode_workspace_bytes(*shape)
    sizes = [ops.decode_workspace_bytes(*shape, dtype=t)
             for t in (torch.bfloat16, torch.float16, torch.float32)]
    assert both == max(sizes) and min(sizes) > 0
    assert ops.decode_workspace_bytes(*shape, -1) == 256
    assert ops.decode_workspace_bytes(shape[0], 5, 2, 64, 8) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_callers_workspace_is_used(dtype):
    dev = "cuda:0"
    n, h, hkv, d, w, bs = 12, 28, 4, 128, 125, 16
    g = torch.Generator(device=dev).manual_seed(1)
    pool = torch.randn(2, w, hkv, bs, d, generator=g, device=dev).to(dtype)
    table = torch.arange(w, dtype=torch.int32, device=dev).repeat(n, 1)
    lens = torch.tensor([1999 - 31 * i for i in range(n)], dtype=torch.int32, device=dev)
    q = torch.randn(n, h, d, generator=g, device=dev).to(dtype)
    ws = ops.decode_workspace(ops.decode_workspace_bytes(n, h, hkv, d, w, bs), dev)
    out = torch.empty_like(q)
    for _ in range(2):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        ops.paged_decode(q, pool, table, lens, d ** -0.5, h, hkv, d, out=out, workspace=ws)
        assert torch.cuda.max_memory_allocated() == before
