"""The vector kernel of the recurrent forward: a decode step, the lengths around its batches of 8 steps and around the
switches to the matrix-core kernels (32 steps; 64 at head dimension 256), against the fp64 oracle."""
import numpy as np
import pytest
import torch

from oracle import gla_oracle as O
from tests.util import assert_plain, check_recurrent_outputs, gpu_inputs, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 7, 8, 17, 32, 33])
@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_few_steps(dtype, D, T):
    from gla_jax_amd import recurrent_gla
    reverse = T % 2 == 1
    (h0, g, v, k, q), dev = gpu_inputs(2, T, 3, D, 1.0, seed=D + T, dtype=dtype)
    hT, out = recurrent_gla(*dev, reverse=reverse)
    flip = (lambda a: a[:, ::-1]) if reverse else (lambda a: a)
    eh, eo = O.recurrent_gla_naive(h0, *(np.ascontiguousarray(flip(a)) for a in (g, v, k, q)))
    check_recurrent_outputs(dtype, (None,) * 5 + (eh, flip(eo)), hT, out)


@pytest.mark.parametrize("D,T", [(64, 1), (128, 5), (256, 64), (256, 65)])
def test_float_state_beside_bf16_rows(D, T):
    """A serving loop carries the state in float32: it is neither rounded on the way in nor on the way out."""
    from gla_jax_amd import recurrent_gla
    (h0, g, v, k, q), dev = gpu_inputs(1, T, 2, D, 3.0, seed=D, dtype=torch.bfloat16)
    h0 = np.random.default_rng(5).standard_normal(h0.shape).astype(np.float32)
    hT, _ = recurrent_gla(to_dev(h0, torch.float32), *dev[1:])
    assert hT.dtype == torch.float32
    assert_plain("hidden_final", to_np(hT), O.recurrent_gla_naive(h0, g, v, k, q)[0], 1e-4)


@pytest.mark.parametrize("D", [16, 64, 128, 256])
def test_values_that_are_not_finite_stay_in_their_column(D):
    """A NaN of the values spoils its column from its step on, an infinite state its column, and a gate of minus infinity
    forgets its row; everything else keeps its bits."""
    from gla_jax_amd import recurrent_gla
    T = 20
    _, dev = gpu_inputs(2, T, 3, D, 1.0, seed=D, dtype=torch.float32)
    dev[1][1, 11, 2, 4] = float("-inf")
    hT, out = recurrent_gla(*dev)
    assert bool(hT.isfinite().all()) and bool(out.isfinite().all())
    gone = [t.clone() for t in dev]                     # what lies in that row before is of no account
    gone[3][1, :11, 2, 4], gone[0][1, 2, 4] = 0.0, 0.0
    ghT, gout = recurrent_gla(*gone)
    assert torch.equal(ghT, hT) and torch.equal(gout[1, 11:], out[1, 11:])

    dev[2][0, 9, 1, 5] = float("nan")
    dev[0][0, 2, 3, 7] = float("inf")
    bad_hT, bad_out = recurrent_gla(*dev)
    want_hT, want_out = hT.clone(), out.clone()
    want_out[0, 9:, 1, 5], want_hT[0, 1, :, 5] = float("nan"), float("nan")
    keep = torch.ones(2, 3, D, dtype=torch.bool, device="cuda")
    keep[0, 2, 7] = False                               # this column's outputs are infinite
    assert not bool(bad_out[0, :, 2, 7].isfinite().any()) and bool(bad_hT[0, 2, 3, 7].isinf())
    keep_rows = torch.ones(2, 3, D, D, dtype=torch.bool, device="cuda")
    keep_rows[0, 2, 3, 7] = False
    same = lambda a, b: bool(((a == b) | (a.isnan() & b.isnan())).all())
    assert same(bad_out.transpose(0, 1)[:, keep], want_out.transpose(0, 1)[:, keep])
    assert same(bad_hT[keep_rows], want_hT[keep_rows])
