"""recurrent_gla in segments that do not divide the length: the last segment (and the last piece of the lean passes, which
can then be a segment's only one) is shorter, down to one step.  Against the fp64 oracle under the usual bounds."""
import numpy as np
import pytest
import torch

from oracle import gla_oracle as O
from tests.util import check_recurrent_outputs, cotangents, gpu_inputs, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,T,H,D,reverse", [
    (torch.bfloat16, 1, 1021, 2, 64, False),      # 7 x 128 + 125
    (torch.bfloat16, 1, 897, 2, 64, True),        # 7 x 128 + 1
    (torch.bfloat16, 1, 321, 1, 128, True),       # 5 x 64 + 1
    (torch.bfloat16, 2, 449, 2, 128, False),
    (torch.bfloat16, 1, 700, 1, 256, True),
    (torch.bfloat16, 4, 1153, 32, 128, False),    # two segments of 640 and 513 steps, lean pieces of 320: 4
    (torch.bfloat16, 4, 1601, 16, 128, True),     # lean passes: 512, 512, 512, 65 in pieces of 256: 7
    (torch.bfloat16, 2, 517, 1, 32, False),
    (torch.float32, 1, 645, 1, 64, True),
    (torch.float32, 1, 513, 1, 256, False),
    (torch.float32, 1, 449, 2, 128, True),        # 7 x 64 + 1
])
def test_uneven_segments_match_oracle(dtype, B, T, H, D, reverse):
    from gla_jax_amd import _lib, recurrent_gla
    dt = _lib.GLA_BF16 if dtype == torch.bfloat16 else _lib.GLA_F32
    assert _lib.load().gla_recurrent_bwd_workspace_bytes(B, T, H, D, D, dt) > 0
    (h0, g, v, k, q), dev = gpu_inputs(B, T, H, D, 3.0, seed=T, dtype=dtype)
    g = g.copy()
    g[:, 127::200] = -200.0
    dev[1] = to_dev(g, torch.float32)
    dhT, dout = cotangents(h0, v, 5, dtype)
    dev = [t.clone().requires_grad_(True) for t in dev]
    hT, out = recurrent_gla(*dev, reverse=reverse)
    grads = torch.autograd.grad((hT, out), dev, (to_dev(dhT, hT.dtype), to_dev(dout, dtype)))
    if B * H >= 16:         # many sequences: the C restatement (fp64), which walks forward in time
        from oracle import naive_c
        fl = (lambda a: np.ascontiguousarray(a[:, ::-1])) if reverse else (lambda a: a)
        dh0_, dg_, dv_, dk_, dq_, hT_, out_ = naive_c.naive_bwd(h0, fl(g), fl(v), fl(k), fl(q), dhT, fl(dout),
                                                                dtype=np.float64, nthreads=16)
        exp = (dh0_, fl(dg_), fl(dv_), fl(dk_), fl(dq_), hT_, fl(out_))
    else:
        exp = O.recurrent_gla_naive_grad(h0, g, v, k, q, dhT, dout, reverse=reverse)
    check_recurrent_outputs(dtype, exp, hT, out, grads)
