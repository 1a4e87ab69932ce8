"""chunk_gla at lengths that the tile does not divide: the last tile is filled up with zeros.  Every tail of every tile that
the choice of tiles reaches, against the fp64 oracle under the usual bounds."""
import pytest
import torch

from tests.util import check_chunk_outputs, cotangents, gpu_inputs, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,T,H,D,shift", [
    (torch.bfloat16, 2, 1056, 8, 128, 5.0),       # 128-token tiles, tails of 32, 64 and 96 tokens
    (torch.bfloat16, 2, 1088, 8, 128, 0.0),
    (torch.bfloat16, 2, 1120, 8, 128, -2.0),      # (every sub-block takes the hard-gate path)
    (torch.bfloat16, 1, 288, 2, 128, 5.0),        # 64-token tiles, a tail of 32
    (torch.bfloat16, 1, 288, 2, 64, -2.0),
    (torch.bfloat16, 1, 4128, 1, 64, 3.0),        # 128-token tiles
    (torch.bfloat16, 1, 2080, 1, 32, 3.0),
    (torch.bfloat16, 1, 2144, 1, 16, 3.0),
    (torch.bfloat16, 1, 288, 1, 256, 3.0),
    (torch.float32, 1, 1056, 1, 64, 3.0),         # 64-token tiles, a tail of 32
    (torch.float32, 1, 1056, 1, 32, 0.0),
    (torch.float32, 1, 1056, 1, 16, 3.0),
    (torch.bfloat16, 1, 608, 2, 32, 3.0),         # 64-token tiles, a tail of 32
    (torch.bfloat16, 1, 608, 2, 16, -2.0),
    # many short sequences: one tile of 32 or 64 tokens each, or of 32 that divides them
    (torch.bfloat16, 33, 32, 8, 64, 3.0),
    (torch.bfloat16, 17, 64, 16, 128, 3.0),
    (torch.bfloat16, 6, 160, 16, 32, 3.0),
    (torch.float32, 33, 32, 8, 64, 3.0),
    (torch.float32, 6, 160, 16, 64, 0.0),
])
def test_last_tile_filled_up_with_zeros(dtype, B, T, H, D, shift):
    from gla_jax_amd import chunk_gla
    arrs, dev = gpu_inputs(B, T, H, D, shift, seed=T + D, dtype=dtype)
    dhT, dout = cotangents(arrs[0], arrs[2], 3, dtype)
    dev = [t.clone().requires_grad_(True) for t in dev]
    hT, out = chunk_gla(*dev, 32)
    grads = torch.autograd.grad((hT, out), dev, (to_dev(dhT, dtype), to_dev(dout, dtype)))
    check_chunk_outputs(dtype, arrs, 32, hT, out, grads, dhT, dout)


@pytest.mark.parametrize("BH,T", [(1, 32 * 15), (1, 64 * 17), (64, 128 * 23)])
def test_scan_over_chunks_with_a_last_batch_that_is_not_full(BH, T):
    """Chunk counts around the scan's batches of 8 and 16: with a zero key every state is the initial one times the decay."""
    from gla_jax_amd import chunk_gla
    D = 32
    _, (h0, g, v, k, q) = gpu_inputs(1, T, BH, D, 5.0, seed=T, dtype=torch.float32)
    g = g / T
    hT, out = chunk_gla(h0, g, v, torch.zeros_like(k), q, 32)
    L = g.double().cumsum(1)
    assert torch.allclose(hT.double(), h0.double() * L[:, -1].exp()[..., None], rtol=1e-5, atol=1e-5)
    want = (q.double() * L.exp()).permute(0, 2, 1, 3) @ h0.double()
    assert torch.allclose(out.double().permute(0, 2, 1, 3), want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("T,shift", [(2048, 3.0), (2080, -2.0)])
def test_float_data_at_128_features_on_64_token_tiles(T, shift):
    from gla_jax_amd import chunk_gla
    dtype = torch.float32
    arrs, dev = gpu_inputs(1, T, 1, 128, shift, seed=T, dtype=dtype)
    dhT, dout = cotangents(arrs[0], arrs[2], 4, dtype)
    dev = [t.clone().requires_grad_(True) for t in dev]
    hT, out = chunk_gla(*dev, 32)
    grads = torch.autograd.grad((hT, out), dev, (to_dev(dhT, dtype), to_dev(dout, dtype)))
    check_chunk_outputs(dtype, arrs, 32, hT, out, grads, dhT, dout)


def _clean_and_filled(dtype, B, T, H, D, full, poison=None):
    """Outputs and gradients of a call of T tokens, and of the same call with zeros up to `full` tokens."""
    from gla_jax_amd import chunk_gla
    arrs, dev = gpu_inputs(B, T, H, D, 3.0, seed=T + D, dtype=dtype)
    dhT, dout = (to_dev(t, dtype) for t in cotangents(arrs[0], arrs[2], 5, dtype))
    results = []
    for n in (T, full):
        args = [dev[0].clone()] + [torch.nn.functional.pad(t, (0, 0, 0, 0, 0, n - T)) for t in dev[1:]]
        if poison is not None:
            poison(args)
        args = [t.requires_grad_(True) for t in args]
        outs = chunk_gla(*args, 32)
        grads = torch.autograd.grad(outs, args, (dhT, torch.nn.functional.pad(dout, (0, 0, 0, 0, 0, n - T))))
        results.append([outs[0], grads[0]] + [t[:, :T] for t in (outs[1],) + grads[1:]])
    return results


# (128-token tiles; at 256 features as two passes of 128 with float results)
@pytest.mark.parametrize("dtype,B,T,H,D,full", [
    (torch.bfloat16, 2, 1056, 8, 256, 1152),
    (torch.bfloat16, 2, 1120, 8, 256, 1152),
    (torch.bfloat16, 2, 1056, 8, 128, 1152),
    (torch.float32, 2, 2080, 2, 128, 2112),
])
def test_tail_is_what_a_caller_would_fill_up(dtype, B, T, H, D, full):
    for got, want in zip(*_clean_and_filled(dtype, B, T, H, D, full)):
        assert torch.equal(got, want)


# (the workspace that head dimension 256 needs beside its passes' own makes their tiles wider than the passes would choose by
# themselves: 128 for 64, and 64 for 32)
@pytest.mark.parametrize("dtype,B,T,H,full", [(torch.bfloat16, 3, 288, 16, 384), (torch.float32, 3, 160, 16, 192)])
def test_passes_of_256_features_take_the_tile_of_the_whole_call(dtype, B, T, H, full):
    for got, want in zip(*_clean_and_filled(dtype, B, T, H, 256, full)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_a_value_that_is_not_finite_in_the_last_tile_stays_with_its_sequence(D, value):
    """One key feature of one token in the filled-up tile: every other (batch, head) pair and the outputs of the tiles before
    keep their bits."""
    def poison(args):
        args[3][0, 1050, 1, 7] = value

    clean = _clean_and_filled(torch.bfloat16, 2, 1056, 16, D, 1152)[0]
    got = _clean_and_filled(torch.bfloat16, 2, 1056, 16, D, 1152, poison)[0]
    others = torch.ones(2, 16, dtype=torch.bool)
    others[0, 1] = False
    for i, (a, b) in enumerate(zip(got, clean)):
        a, b = (a, b) if i < 2 else (a.transpose(1, 2), b.transpose(1, 2))
        assert torch.equal(a[others], b[others])
        if i in (1, 5):          # the gradients of the initial state and of the keys have no key in them
            assert torch.equal(a, b)
        else:
            assert not bool(a[0, 1].isfinite().all())
    assert torch.equal(got[2][0, :1024, 1], clean[2][0, :1024, 1])


def test_short_sequences_do_not_pay_for_a_wide_tile():
    """One tile per sequence: 32 tokens on a tile of 32 take 0.60 of the time of 128 tokens, on a tile of 128 they took 0.78."""
    from gla_jax_amd import chunk_gla
    gen = torch.Generator(device="cuda").manual_seed(1)
    normal = lambda *s: torch.randn(*s, generator=gen, device="cuda")

    def milliseconds(T):
        rows = [normal(128, T, 16, 128).bfloat16() for _ in range(4)]
        h0, gates = normal(128, 16, 128, 128).bfloat16(), torch.nn.functional.logsigmoid(3 + normal(128, T, 16, 128))
        args = [t.requires_grad_(True) for t in (h0, gates, *rows[:3])]
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(3):
                torch.autograd.grad(chunk_gla(*args, 32), args, (h0.detach(), rows[3]))
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert milliseconds(32) < 0.7 * milliseconds(128)
