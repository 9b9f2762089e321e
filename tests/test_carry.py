"""The carry of a chain of single steps is updated in place, so it must never be the caller's own states."""
import pytest
import torch

from flashrnn_amd import make_carry


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 3])
def test_make_carry_returns_memory_of_its_own(dtype, T):
    states = torch.randn(2, 3, T, 2, 32).to(dtype)[:, :, -1:]
    before = states.clone()
    carry = make_carry(states)
    assert carry.dtype == torch.float32 and carry.shape == (2, 3, 2, 32) and carry.is_contiguous()
    assert torch.equal(carry, states[:, :, 0].float())
    carry.add_(1.0)
    assert torch.equal(states, before)
