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
