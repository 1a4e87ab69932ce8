"""Calls that the torch entry points refuse before anything is launched.  The arrays are fake ones that say they lie on a
GPU: what is not refused ends in an error about their missing memory."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from gla_jax_amd import rnn_recursive


@pytest.fixture
def zeros():
    with FakeTensorMode():
        yield lambda *shape, device="cuda:0", dtype=torch.float32: torch.zeros(*shape, device=device, dtype=dtype)


@pytest.mark.parametrize("lead, init", [((3,), (8,)), ((3,), (2, 8)), ((), (7,)), ((3,), (3, 9))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rnn_init_of_another_size(zeros, lead, init, dtype):
    """One pair for a whole batch, or a pair of other sizes: the kernel would read past it."""
    a, kv = zeros(*lead, 5, 8, dtype=dtype), zeros(*lead, 5, 8, 4, dtype=dtype)
    with pytest.raises(AssertionError, match="init"):
        rnn_recursive(a, kv, zeros(*init), zeros(*init, 4))
    with pytest.raises(AssertionError, match="init"):
        rnn_recursive(a, kv, zeros(*lead, 8), zeros(*init, 4))
