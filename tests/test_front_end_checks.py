"""Calls that the torch entry points refuse before anything is launched.  The arrays are fake ones that say they lie on a
GPU: what is not refused ends in an error about their missing memory."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from gla_jax_amd import chunk_gla, cumsum_recursive, recurrent_gla, recurrent_gla_naive, rnn_recursive


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


@pytest.mark.parametrize("odd_one", range(5))
@pytest.mark.parametrize("fn", [lambda *a: chunk_gla(*a, 32), recurrent_gla, lambda *a: recurrent_gla_naive(*a, False)])
def test_arrays_on_different_devices(zeros, fn, odd_one):
    arrays = [zeros(2, 4, 16, 16)] + [zeros(2, 64, 4, 16) for _ in range(4)]
    arrays[odd_one] = zeros(*arrays[odd_one].shape, device="cuda:1")
    with pytest.raises(ValueError, match="device"):
        fn(*arrays)


def test_scan_arrays_on_different_devices(zeros):
    with pytest.raises(ValueError, match="device"):
        cumsum_recursive(zeros(4, 64, 8), 1, init=zeros(4, 8, device="cuda:1"))
    a, kv = zeros(3, 5, 8), zeros(3, 5, 8, 4)
    for args in [(a, zeros(3, 5, 8, 4, device="cuda:1")), (a, kv, zeros(3, 8, device="cuda:1"), zeros(3, 8, 4)),
                 (a, kv, zeros(3, 8), zeros(3, 8, 4, device="cuda:1"))]:
        with pytest.raises(ValueError, match="device"):
            rnn_recursive(*args)
