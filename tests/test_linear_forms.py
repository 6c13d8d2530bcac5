"""layers.linear.Linear is nn.Linear wherever the call is more than its values: under tracing,
function transforms, forward- and reverse-mode differentiation and autocast (on the CPU, where
every call is torch's own), with the parameters and state dict of nn.Linear."""
import copy

import pytest
import torch
import torch.nn as nn
from torch.autograd import forward_ad

from needle_amd import ops
from needle_amd.layers.linear import Linear


@pytest.fixture()
def pair():
    torch.manual_seed(0)
    ours = Linear(64, 32)
    theirs = nn.Linear(64, 32)
    theirs.load_state_dict(ours.state_dict())
    return ours, theirs, torch.randn(5, 64)


def test_values_gradients_and_copies(pair):
    ours, theirs, x = pair
    assert [n for n, _ in ours.named_parameters()] == [n for n, _ in theirs.named_parameters()]
    for shape in ((5, 64), (1, 5, 64), (64,)):
        xs = x[0] if shape == (64,) else x.reshape(shape)
        assert torch.equal(ours(xs), theirs(xs))
    ours(x).sum().backward()
    theirs(x).sum().backward()
    assert torch.equal(ours.weight.grad, theirs.weight.grad)
    assert torch.equal(copy.deepcopy(ours)(x), theirs(x))
    with torch.autocast("cpu", dtype=torch.bfloat16):
        assert ours(x).dtype == torch.bfloat16 and torch.equal(ours(x), theirs(x))


def test_transforms(pair):
    ours, theirs, x = pair
    assert torch.equal(torch.func.vmap(ours)(x), torch.func.vmap(theirs)(x))
    with forward_ad.dual_level():
        d = forward_ad.make_dual(x, torch.ones_like(x))
        a, b = forward_ad.unpack_dual(ours(d)), forward_ad.unpack_dual(theirs(d))
    assert torch.equal(a.tangent, b.tangent)
    assert torch.equal(torch.fx.symbolic_trace(ours)(x), theirs(x))
    assert torch.equal(torch.jit.trace(ours, (x,))(x), theirs(x))


@pytest.mark.parametrize("owner,name", [(torch._C._functorch, "peek_interpreter_stack"),
                                        (torch._C, "_len_torch_dispatch_stack"),
                                        (torch._C, "_len_torch_function_stack"),
                                        (forward_ad, "_current_level")])
def test_a_missing_private_name_means_torchs_own(monkeypatch, owner, name):
    assert ops._plain_call()
    monkeypatch.delattr(owner, name)
    assert not ops._plain_call()
