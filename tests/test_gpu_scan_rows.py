"""cumsum_recursive on rows of 64 columns and more: lengths around a block's rows (128 and 256), a wave's and a lane's, one and
many stretches, columns that do not fill a tile, arrays that are not 16-byte aligned (the kernels for any layout)."""
import pytest
import torch

from gla_jax_amd import cumsum_recursive

pytestmark = pytest.mark.gpu


def reference(x, init, reverse):
    y = x.double().flip(1) if reverse else x.double()
    y = y.cumsum(1) + (0 if init is None else init.double()[:, None])
    return y.flip(1) if reverse else y


@pytest.mark.parametrize("outer,T,inner", [(2, 32, 64), (3, 33, 68), (1, 127, 128), (2, 128, 132), (2, 129, 64), (1, 256, 192),
                                           (2, 257, 128), (1, 511, 260), (3, 1120, 768), (1, 2049, 64), (5, 2100, 1024)])
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("form", ["plain", "init", "unaligned"])
def test_cumsum_of_long_rows(outer, T, inner, reverse, form):
    gen = torch.Generator(device="cuda").manual_seed(T)
    flat = torch.randn(outer * T * inner + 1, generator=gen, device="cuda")
    x = flat[1 if form == "unaligned" else 0:][:outer * T * inner].view(outer, T, inner)
    init = torch.randn(outer, inner, generator=gen, device="cuda") if form == "init" else None
    got = cumsum_recursive(x, 1, init=init, reverse=reverse)
    # a result passes through at most 100 additions (rows of a lane, groups of a block twice, stretches over the groups; four
    # rows per step and a few segments in the other kernels, which hold up to 600 rows at these sizes), each off by 2^-24 of a sum
    # that is at most the sum of magnitudes
    depth = 700 if form == "unaligned" else 100
    bound = depth * 2.0 ** -24 * (x.abs().double().sum(1, keepdim=True) + (0 if init is None else init.abs().double()[:, None]))
    assert bool(((got - reference(x, init, reverse)).abs() <= bound).all())


def test_a_value_that_is_not_finite_stays_behind_its_row():
    x = torch.ones(1, 1000, 64, device="cuda")
    x[0, 300, 5], x[0, 640, 6] = float("inf"), float("nan")
    for reverse in (False, True):
        got, exp = cumsum_recursive(x, 1, reverse=reverse), reference(x, None, reverse)
        assert torch.allclose(got.double(), exp, rtol=0, atol=0, equal_nan=True)
