"""chunk_gla on bf16 data at head dimension 256, whose second pass takes the value-side rows of the other half where they lie and
adds what the first pass left: with one half of the key features empty, `out` and dvalue are those of 128-feature problems, bit
for bit (the sum is with zeros).  Lengths around the edges of the tiles, whole waves without tokens among them."""
import pytest
import torch

from tests.util import gpu_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [32, 96, 128, 160, 288, 416])
@pytest.mark.parametrize("empty", [0, 1])
def test_halves_of_256_features_are_problems_of_128(T, empty):
    from gla_jax_amd import chunk_gla
    B, H = 2, 3
    _, (h0, g, v, k, q) = gpu_inputs(B, T, H, 256, 3.0, seed=T, dtype=torch.bfloat16)
    dout = torch.randn(B, T, H, 256, generator=torch.Generator("cuda").manual_seed(T), device="cuda").bfloat16()
    for t in (k, q):
        t.view(B, T, 2 * H, 128)[:, :, empty::2] = 0
    h0 = torch.zeros_like(h0)

    def run(h0, g, v, k, q, dout):
        args = [t.clone().requires_grad_(True) for t in (h0, g, v, k, q)]
        hT, out = chunk_gla(*args, 32)
        grads = torch.autograd.grad((hT, out), args, (torch.zeros_like(hT), dout))
        return out.detach(), grads[2]

    whole = [t.view(B, T, 2 * H, 128) for t in run(h0, g, v, k, q, dout)]
    rows = [t.reshape(B, T, 2 * H, 128) for t in (g, v, k, q, dout)]
    swapped = [t.view(B, T, H, 2, 128).flip(3).reshape(B, T, 2 * H, 128) for t in (rows[1], rows[4])]
    states = torch.zeros(B, 2 * H, 128, 128, dtype=torch.bfloat16, device="cuda")
    same = run(states, *rows)
    cross = run(states, rows[0], swapped[0], rows[2], rows[3], swapped[1])
    full = 1 - empty
    for got, a, b in zip(whole, same, cross):
        assert torch.equal(got[:, :, full::2], a[:, :, full::2])
        assert torch.equal(got[:, :, empty::2], b[:, :, full::2])
        assert bool(got.abs().amax() > 0)
