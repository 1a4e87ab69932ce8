"""What autograd does around a forward and its backward: saved-tensor hooks, checkpointing, errors."""
import pytest
import torch

from tests.util import gpu_inputs

pytestmark = pytest.mark.gpu

# few sequences of 320 steps: recurrent_gla runs them as segments and hands their states to the backward
NAMES = ["chunk_gla", "recurrent_gla", "recurrent_gla_naive"]


def _bind(name):
    import gla_jax_amd
    return {"chunk_gla": lambda *a: gla_jax_amd.chunk_gla(*a, 32), "recurrent_gla": gla_jax_amd.recurrent_gla,
            "recurrent_gla_naive": lambda *a: gla_jax_amd.recurrent_gla_naive(*a, False)}[name]


def _problem(name, seed, D=64, dtype=torch.bfloat16):
    dev = [t.requires_grad_(True) for t in gpu_inputs(1, 320, 2, D, 3.0, seed=seed, dtype=dtype)[1]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.no_grad():
        outs = _bind(name)(*dev)
    return dev, [torch.randn(o.shape, generator=gen, device="cuda").to(o.dtype) for o in outs]


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("create_graph", [False, True])
def test_saved_tensors_come_back_in_another_layout(name, create_graph):
    fn = _bind(name)
    dev, ct = _problem(name, 41)
    want = torch.autograd.grad(fn(*dev), dev, ct)
    spread = lambda t: torch.stack((t, t), -1)[..., 0]          # the same values, two elements apart
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), spread):
        outs = fn(*dev)
        got = torch.autograd.grad(outs, dev, ct, create_graph=create_graph)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", NAMES)
def test_saved_tensors_that_come_back_as_others_are_refused(name):
    fn = _bind(name)
    dev, ct = _problem(name, 42)
    for other in (lambda t: t.cpu(), lambda t: t.to(torch.float64), lambda t: t.flatten()[:-16]):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, other):
            outs = fn(*dev)
            with pytest.raises(RuntimeError, match="saved-tensor hook"):
                torch.autograd.grad(outs, dev, ct)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("use_reentrant", [False, True])
def test_checkpoint(name, use_reentrant):
    from torch.utils.checkpoint import checkpoint
    fn = _bind(name)
    dev, ct = _problem(name, 43)
    want = torch.autograd.grad(fn(*dev), dev, ct)
    args = [t.detach().clone().requires_grad_(True) for t in dev]
    torch.autograd.backward(checkpoint(fn, *args, use_reentrant=use_reentrant), ct)
    for a, b in zip(args, want):
        assert torch.equal(a.grad, b)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("grad", [False, True])
def test_traced_call_computes_on_new_inputs(name, grad):
    """torch.jit.trace records the call itself, not the buffers it fills."""
    fn = _bind(name)
    dev, ct = _problem(name, 44)
    new = [t.detach().clone().requires_grad_(grad) for t in _problem(name, 45)[0]]
    traced = torch.jit.trace(fn, tuple(t.detach().requires_grad_(grad) for t in dev), check_trace=False)
    got, want = traced(*new), fn(*new)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    if grad:
        for a, b in zip(torch.autograd.grad(got, new, ct), torch.autograd.grad(want, new, ct)):
            # (the traced forward hands no segment states to its backward, which forms them again to the same bits)
            assert torch.equal(a, b)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("create_graph", [False, True])
def test_status_of_a_backward_reaches_the_caller(name, create_graph):
    """A cotangent that is dense but not 16-byte aligned is refused by the library; the status arrives as it does in a forward."""
    from gla_jax_amd._lib import GlaError
    fn = _bind(name)
    dev, ct = _problem(name, 46)
    outs = fn(*dev)
    shifted = torch.zeros(ct[1].numel() + 1, device="cuda", dtype=ct[1].dtype)[1:].view(ct[1].shape)
    with pytest.raises(GlaError) as e:
        torch.autograd.grad(outs[1], dev, shifted, create_graph=create_graph)
    assert e.value.status == -6
    shifted = torch.zeros(dev[4].numel() + 1, device="cuda", dtype=dev[4].dtype)[1:].view(dev[4].shape)
    with pytest.raises(GlaError) as e:
        fn(*dev[:4], shifted)
    assert e.value.status == -6
