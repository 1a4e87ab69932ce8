"""recurrent_gla on bf16 data at head dimension 256, whose second pass takes the value-side rows of the other half where they lie
and adds what the first pass left: lengths next to the edges of the 64-step blocks, whole sequences and segments of them (an
fp32 state beside the bf16 arrays included), against the fp64 oracle."""
import pytest
import torch

from oracle import gla_oracle as O
from tests.util import check_recurrent_outputs, cotangents, gpu_inputs, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [65, 127, 129, 320])
@pytest.mark.parametrize("reverse", [False, True])
def test_passes_of_256_features(T, reverse):
    from gla_jax_amd import recurrent_gla
    dtype = torch.bfloat16
    (h0, g, v, k, q), dev = gpu_inputs(2, T, 3, 256, 3.0, seed=T, dtype=dtype)
    dhT, dout = cotangents(h0, v, 11, dtype)
    dev = [t.clone().requires_grad_(True) for t in dev]
    hT, out = recurrent_gla(*dev, reverse=reverse)
    grads = torch.autograd.grad((hT, out), dev, (to_dev(dhT, dtype), to_dev(dout, dtype)))
    exact = O.recurrent_gla_naive_grad(h0, g, v, k, q, dhT, dout, reverse=reverse)
    check_recurrent_outputs(dtype, exact, hT, out, grads)
    wide = [dev[0].detach().float(), *[t.detach() for t in dev[1:]]]
    assert torch.equal(recurrent_gla(*wide, reverse=reverse)[1], out.detach())


@pytest.mark.parametrize("T", [48, 65, 192, 320])          # 320: as segments, their states from the lean passes
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("hard", [(0,), (1,), (2,), (3,), (0, 3), (0, 1, 2, 3)])
def test_hard_gates_in_some_quarters_of_256_features(T, reverse, hard):
    """A wave has a quarter of the key features and decides for itself whether its gates are hard.  Its part of dq then waits in the
    pass's own q*dq array and its part of dk in the exchange buffer, and what the first pass left is added behind them."""
    from gla_jax_amd import recurrent_gla, recurrent_gla_naive
    dtype = torch.bfloat16
    (h0, g, v, k, q), dev = gpu_inputs(1, T, 2, 256, 3.0, seed=T, dtype=dtype)
    g = g.copy()
    for quarter in hard:
        g[:, 3 + quarter::11, :, 64 * quarter:64 * quarter + 64] = -60.0
    dev[1] = to_dev(g, torch.float32)
    dhT, dout = cotangents(h0, v, 11, dtype)
    exact = O.recurrent_gla_naive_grad(h0, g, v, k, q, dhT, dout, reverse=reverse)
    check_recurrent_outputs(dtype, exact, *recurrent_gla_naive(*dev, reverse=reverse), out_fp32=True)
    dev = [t.clone().requires_grad_(True) for t in dev]
    hT, out = recurrent_gla(*dev, reverse=reverse)
    grads = torch.autograd.grad((hT, out), dev, (to_dev(dhT, dtype), to_dev(dout, dtype)))
    check_recurrent_outputs(dtype, exact, hT, out, grads)
