"""Function transforms around the torch entry points: several vector-Jacobian products of one forward."""
import pytest
import torch

from tests.util import gpu_inputs

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, D, seed, dtype=torch.bfloat16):
    return gpu_inputs(B, T, H, D, 3.0, seed=seed, dtype=dtype)[1]


def _cotangents(n, outs, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(n, *o.shape, generator=gen, device="cuda").to(o.dtype) for o in outs]


def _bind(name):
    import gla_jax_amd
    return {"chunk_gla": lambda *a: gla_jax_amd.chunk_gla(*a, 32), "recurrent_gla": gla_jax_amd.recurrent_gla,
            "recurrent_gla_naive": lambda *a: gla_jax_amd.recurrent_gla_naive(*a, False)}[name]


# (1, 256, 64, 64): 64-token tiles for one batch entry, 128-token tiles for three: another layout of the states
@pytest.mark.parametrize("name, shape", [("chunk_gla", (2, 96, 2, 64)), ("chunk_gla", (1, 256, 64, 64)),
                                         ("chunk_gla", (1, 64, 1, 256)), ("recurrent_gla", (2, 96, 2, 64)),
                                         ("recurrent_gla_naive", (1, 40, 2, 32))])
def test_mapped_cotangents_of_one_forward(name, shape):
    fn, dev = _bind(name), _inputs(*shape, seed=31)
    outs, vjp = torch.func.vjp(fn, *dev)
    ct = _cotangents(3, outs, 32)
    got = torch.func.vmap(lambda *c: vjp(c))(*ct)
    only_out = torch.func.vmap(lambda c: vjp((torch.zeros_like(outs[0]), c)))(ct[1])
    for i in range(3):
        for a, b in zip(got, vjp((ct[0][i], ct[1][i]))):
            assert torch.equal(a[i], b)
        for a, b in zip(only_out, vjp((torch.zeros_like(outs[0]), ct[1][i]))):
            assert torch.equal(a[i], b)


@pytest.mark.parametrize("name", ["chunk_gla", "recurrent_gla"])
def test_mapped_cotangents_of_a_mapped_forward(name):
    """One mapped axis of the arrays, another of the cotangents, inside and outside of each other."""
    fn, dev = _bind(name), _inputs(4, 64, 2, 64, seed=33)
    dev = [t.unflatten(0, (2, 2)) for t in dev]
    outs = fn(*dev)
    ct = _cotangents(3, outs, 34)
    want = []
    for i in range(3):
        args = [t.clone().requires_grad_(True) for t in dev]
        want.append(torch.autograd.grad(fn(*args), args, [c[i] for c in ct]))

    def products(*a):                    # the forward inside the mapped axis, its cotangents mapped within
        arrays, c = a[:5], a[5:]
        _, vjp = torch.func.vjp(fn, *arrays)
        return torch.func.vmap(lambda *x: vjp(x))(*c)

    inner = torch.func.vmap(products, in_dims=(0,) * 5 + (1, 1), out_dims=1)(*dev, *ct)
    _, vjp = torch.func.vjp(torch.func.vmap(fn), *dev)
    outer = torch.func.vmap(lambda *x: vjp(x))(*ct)
    # an initial state mapped alone: the rows are shared, the states are not
    h0 = dev[0]
    _, vjp = torch.func.vjp(torch.func.vmap(fn, in_dims=(0, None, None, None, None)), h0, *(t[0] for t in dev[1:]))
    shared = vjp(tuple(c[0] for c in ct))
    for i in range(3):
        for a, b, w in zip(inner, outer, want[i]):
            assert torch.equal(a[i], w) and torch.equal(b[i], w)
    args = [h0.clone().requires_grad_(True)] + [t[0].clone().requires_grad_(True) for t in dev[1:]]
    parts = [fn(args[0][m], *args[1:]) for m in range(2)]
    each = torch.autograd.grad(parts[0] + parts[1], args, [c[0][m] for m in range(2) for c in ct])
    assert torch.equal(shared[0], each[0])
    for a, b in zip(shared[1:], each[1:]):
        # the sum over the mapped axis is formed in the element type by both, from the same two terms
        assert torch.equal(a, b) or (a.float() - b.float()).norm() <= 2 ** -8 * b.float().norm()


@pytest.mark.parametrize("name, D", [("chunk_gla", 64), ("recurrent_gla", 64), ("recurrent_gla", 8), ("recurrent_gla_naive", 128)])
@pytest.mark.parametrize("create_graph", [False, True])
def test_mapped_backward_of_a_plain_forward(name, D, create_graph):
    """The transform is active in the backward alone.  Sequences of 320 steps run as segments in recurrent_gla."""
    fn = _bind(name)
    for shape in ((2, 64, 2, D), (1, 320, 1, D)):
        dev = [t.requires_grad_(True) for t in _inputs(*shape, seed=35)]
        outs = fn(*dev)
        ct = _cotangents(3, outs, 36)
        grad = lambda y, *c: torch.autograd.grad(y, dev, c, retain_graph=True, create_graph=create_graph)
        got = torch.func.vmap(lambda a, b: grad(outs, a, b))(*ct)
        only_out = torch.func.vmap(lambda b: grad(outs[1], b))(ct[1])
        for i in range(3):
            for mapped, single in ((got, grad(outs, ct[0][i], ct[1][i])), (only_out, grad(outs[1], ct[1][i]))):
                for a, b in zip(mapped, single):
                    if shape[1] == 64 or name == "chunk_gla":
                        assert torch.equal(a[i], b)
                    # three times the sequences are cut into other segments: sums in another order, rounded once to bf16
                    assert (a[i].float() - b.float()).norm() <= 2 ** -8 * b.float().norm()


@pytest.mark.parametrize("name", ["chunk_gla", "recurrent_gla"])
def test_batched_cotangents_of_the_older_mapping_are_refused(name):
    dev = [t.requires_grad_(True) for t in _inputs(1, 64, 1, 64, seed=37)]
    outs = _bind(name)(*dev)
    with pytest.raises(NotImplementedError, match="torch.func.vmap"):
        torch.autograd.grad(outs, dev, _cotangents(3, outs, 38), is_grads_batched=True)
