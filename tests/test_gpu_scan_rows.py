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


# 256 stretches (of 256 rows) are added up, more of them (of 128) scanned, 66000 in turn as stretches of stretches
@pytest.mark.parametrize("outer,T,inner", [(1, 65536, 64), (1, 65537, 64), (2, 40000, 132), (1, 128 * 66000 + 3, 64),
                                           (1, 257, 65536 * 4)])    # (256 MB read by the kernel for any layout)
@pytest.mark.parametrize("reverse", [False, True])
def test_cumsum_of_long_axes(outer, T, inner, reverse):
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(outer, T, inner, generator=gen, device="cuda")
    init = torch.randn(outer, inner, generator=gen, device="cuda")
    got = cumsum_recursive(x, 1, init=init, reverse=reverse)
    # a lane's rows and a block's groups three times over, and 256 stretches added up by 8 or 16 groups: at most 150 additions
    step = 44 if T > 1000 else inner
    for c in range(0, inner, step):          # (a few columns at a time: the reference holds 64 bits)
        part = x[..., c:c + step]
        bound = 150 * 2.0 ** -24 * (part.abs().double().sum(1, keepdim=True) + init[:, None, c:c + step].abs().double())
        assert bool(((got[..., c:c + step] - reference(part, init[:, c:c + step], reverse)).abs() <= bound).all())


def test_cumsum_grows_with_its_axis():
    """Four times the rows take four times as long, not sixteen (the sums of 32768 stretches added up by each of them)."""
    def seconds(T):
        x = torch.zeros(1, T, 64, device="cuda")
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            cumsum_recursive(x, 1)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert seconds(1 << 22) < 8 * seconds(1 << 20)


@pytest.mark.parametrize("shape,axis", [((2, 1000, 128), 1), ((3, 40, 64), 1), ((70000, 33), 0), ((70000, 3, 2), 1)])
def test_converted_arrays_take_the_same_way(shape, axis):
    """16-bit and strided arrays are converted first: the bits of a call with the converted ones."""
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(*shape, generator=gen, device="cuda")
    init = torch.randn(*shape[:axis], *shape[axis + 1:], generator=gen, device="cuda").bfloat16()
    spread = torch.stack((x, x), -1)[..., 0]
    for reverse in (False, True):
        assert torch.equal(cumsum_recursive(spread, axis, reverse=reverse), cumsum_recursive(x, axis, reverse=reverse))
        low = x.bfloat16()
        want = cumsum_recursive(low.float(), axis, init=init.float(), reverse=reverse)
        assert torch.equal(cumsum_recursive(low, axis, init=init, reverse=reverse), want.bfloat16())


def test_a_value_that_is_not_finite_stays_behind_its_row():
    x = torch.ones(1, 1000, 64, device="cuda")
    x[0, 300, 5], x[0, 640, 6] = float("inf"), float("nan")
    for reverse in (False, True):
        got, exp = cumsum_recursive(x, 1, reverse=reverse), reference(x, None, reverse)
        assert torch.allclose(got.double(), exp, rtol=0, atol=0, equal_nan=True)
