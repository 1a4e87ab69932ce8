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
