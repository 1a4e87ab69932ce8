"""The chunk states that a backward call is handed are those of a forward over the same batch: the kernels read them by
address.  The launches are replaced by records of what they were asked for, so no GPU is needed."""
import pytest
import torch

from gla_jax_amd import _lib, gla


class _Records:
    """The library with its two chunk launches replaced; sizes come from the real one."""

    def __init__(self, real):
        self.real, self.formed, self.checked = real, {}, 0

    def __getattr__(self, name):
        return getattr(self.real, name)

    def gla_chunk_fwd(self, stream, B, *rest):
        self.formed[rest[14]] = B                # the residual's address
        return 0

    def gla_chunk_bwd(self, stream, B, *rest):
        assert self.formed[rest[11]] == B
        self.checked += 1
        return 0


@pytest.fixture
def records(monkeypatch):
    r = _Records(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: r)
    monkeypatch.setattr(gla, "_stream", lambda: None)
    return r


def _arrays(lead, T=64, H=1, D=32):
    return [torch.zeros(*lead, H, D, D)] + [torch.zeros(*lead, T, H, D) for _ in range(4)]


def test_mapped_cotangents(records):
    dev = _arrays((2,))
    outs, vjp = torch.func.vjp(lambda *a: gla._ChunkGLA.apply(*a, 32)[:2], *dev)
    got = torch.func.vmap(lambda *c: vjp(c))(*(torch.zeros(3, *o.shape) for o in outs))
    assert records.checked == 3 and got[1].shape == (3,) + dev[1].shape


def test_mapped_arrays(records):
    dev = _arrays((5, 2))
    one = lambda *a: gla._ChunkGLA.apply(*a, 32)[:2]
    outs, vjp = torch.func.vjp(torch.func.vmap(one), *dev)
    got = vjp(tuple(torch.zeros_like(o) for o in outs))
    assert records.formed and set(records.formed.values()) == {10}
    assert records.checked == 1 and all(a.shape == b.shape for a, b in zip(got, dev))


def test_initial_state_mapped_alone(records):
    dev = _arrays((5, 2))[:1] + _arrays((2,))[1:]
    one = lambda *a: gla._ChunkGLA.apply(*a, 32)[:2]
    outs, vjp = torch.func.vjp(torch.func.vmap(one, in_dims=(0, None, None, None, None)), *dev)
    got = vjp(tuple(torch.zeros_like(o) for o in outs))
    assert set(records.formed.values()) == {10}
    assert records.checked == 1 and all(a.shape == b.shape for a, b in zip(got, dev))
