"""recurrent_gla on bf16 data at head dimension 128, where two waves share a 16-step sub-block: lengths around the edges of
the 64-step blocks and of their sub-blocks, gates that are mild in one half of the key features and hard in the other (each
wave decides for its own half), against the fp64 oracle."""
import pytest
import torch

from oracle import gla_oracle as O
from tests.util import check_recurrent_outputs, cotangents, gpu_inputs, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [33, 48, 63, 64, 65, 80, 127, 129, 192])
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("hard", ["", "first half", "second half"])
def test_two_waves_per_sub_block(T, reverse, hard):
    from gla_jax_amd import recurrent_gla
    dtype = torch.bfloat16
    arrs, dev = gpu_inputs(1, T, 2, 128, 3.0, seed=T, dtype=dtype)
    h0, g, v, k, q = arrs
    if hard:
        g = g.copy()
        g[:, 3::11, :, :64 if hard == "first half" else 128][..., -64:] = -60.0
        dev[1] = to_dev(g, torch.float32)
    dhT, dout = cotangents(h0, v, 11, dtype)
    dev = [t.clone().requires_grad_(True) for t in dev]
    hT, out = recurrent_gla(*dev, reverse=reverse)
    grads = torch.autograd.grad((hT, out), dev, (to_dev(dhT, dtype), to_dev(dout, dtype)))
    exact = O.recurrent_gla_naive_grad(h0, g, v, k, q, dhT, dout, reverse=reverse)
    check_recurrent_outputs(dtype, exact, hT, out, grads)
