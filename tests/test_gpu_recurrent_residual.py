"""recurrent_gla in segments with the forward's states handed to the backward: the same bits as a backward that forms them."""
import pytest
import torch

from gla_jax_amd import _lib, recurrent_gla
from tests.util import cotangents, gpu_inputs, to_dev


# one size per way the segments come about: lean passes in one and two pieces, a full first pass, head dimension 256, an
# fp32 output beside bf16 data, a last segment that is shorter, both directions
@pytest.mark.gpu
@pytest.mark.parametrize("B,T,H,D,dtype,out_fp32,reverse", [
    (1, 1021, 8, 64, torch.bfloat16, False, False),
    (1, 1021, 8, 64, torch.bfloat16, True, True),
    (2, 2050, 16, 128, torch.bfloat16, False, True),
    (1, 230, 2, 128, torch.bfloat16, False, False),
    (1, 700, 2, 256, torch.bfloat16, False, False),
    (1, 777, 3, 64, torch.float32, False, True),
    (1, 512, 4, 32, torch.bfloat16, True, False),
])
def test_backward_with_the_forwards_states_gives_the_same_bits(B, T, H, D, dtype, out_fp32, reverse):
    lib = _lib.load()
    arrs, (h0, g, v, k, q) = gpu_inputs(B, T, H, D, 3.0, seed=11, dtype=dtype)
    dhT, dout = (to_dev(t, dtype) for t in cotangents(arrs[0], arrs[2], 11, dtype))
    dout = dout.to(torch.float32 if out_fp32 else dtype).contiguous()
    code = lambda t: _lib.GLA_F32 if t.dtype == torch.float32 else _lib.GLA_BF16
    head = (torch.cuda.current_stream().cuda_stream, B, T, H, D, D, code(v), code(h0), code(dout), int(reverse))
    sizes = (B, T, H, D, D, code(v))
    nbytes = lambda n: torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    nf, nb, nr = lib.gla_recurrent_fwd_workspace_bytes(*sizes), lib.gla_recurrent_bwd_workspace_bytes(*sizes), \
        lib.gla_recurrent_residual_bytes(*sizes)
    assert 0 < nr <= nf
    p = lambda *ts: [t.data_ptr() for t in ts]

    def both(residual):
        hT, out = torch.empty_like(h0), torch.empty_like(dout)
        ws = nbytes(nf)
        _lib.check("fwd", lib.gla_recurrent_fwd_res(*head, *p(h0, g, v, k, q, hT, out), residual, ws.data_ptr(), nf))
        grads = [torch.empty_like(t) for t in (h0, g, v, k, q)]
        ws = nbytes(nb)
        _lib.check("bwd", lib.gla_recurrent_bwd_res(*head, *p(h0, g, v, k, q, hT, dhT, dout, *grads), residual, ws.data_ptr(), nb))
        torch.cuda.synchronize()
        return [hT, out] + grads

    res = nbytes(nr)
    for got, ref in zip(both(res.data_ptr()), both(None)):
        assert torch.equal(got, ref)


@pytest.mark.gpu
def test_states_kept_for_the_backward_serve_several_backward_passes():
    arrs, dev = gpu_inputs(1, 1021, 8, 64, 3.0, seed=12, dtype=torch.bfloat16)
    dev = [t.clone().requires_grad_(True) for t in dev]
    dhT, dout = (to_dev(t, torch.bfloat16) for t in cotangents(arrs[0], arrs[2], 12, torch.bfloat16))
    outs = recurrent_gla(*dev)
    first = torch.autograd.grad(outs, dev, [dhT, dout], retain_graph=True)
    recurrent_gla(*[t.detach() * 0 for t in dev])      # another call between the two
    for a, b in zip(first, torch.autograd.grad(outs, dev, [dhT, dout])):
        assert torch.equal(a, b)
    grads = torch.autograd.grad(recurrent_gla(*dev), dev, [dhT, dout], create_graph=True)
    for a, b in zip(first, grads):
        assert torch.equal(a, b)
    with pytest.raises(NotImplementedError, match="second-order"):
        grads[0].float().sum().backward()


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,H,D,dtype,out_fp32", [(1, 256, 8, 16, torch.bfloat16, True), (2, 295, 4, 32, torch.float32, False),
                                                    (1, 300, 2, 64, torch.float32, False)])
def test_forward_alone_runs_two_segments_whole(B, T, H, D, dtype, out_fp32):
    """Where the pass before the segments is a full one: the bits of the call without a workspace."""
    lib = _lib.load()
    _, (h0, g, v, k, q) = gpu_inputs(B, T, H, D, 3.0, seed=13, dtype=dtype)
    code = _lib.GLA_F32 if dtype == torch.float32 else _lib.GLA_BF16
    nf = lib.gla_recurrent_fwd_workspace_bytes(B, T, H, D, D, code)
    assert nf > 0
    head = (torch.cuda.current_stream().cuda_stream, B, T, H, D, D, code, code, _lib.GLA_F32 if out_fp32 else code, 0)
    results = []
    for ws in (None, torch.empty(nf, dtype=torch.uint8, device="cuda")):
        hT, out = torch.empty_like(h0), torch.empty_like(v, dtype=torch.float32 if out_fp32 else dtype)
        arrays = [t.data_ptr() for t in (h0, g, v, k, q, hT, out)]
        _lib.check("fwd", lib.gla_recurrent_fwd(*head, *arrays) if ws is None else
                   lib.gla_recurrent_fwd_ws(*head, *arrays, ws.data_ptr(), nf))
        results.append((hT, out))
    for a, b in zip(*results):
        assert torch.equal(a, b)
