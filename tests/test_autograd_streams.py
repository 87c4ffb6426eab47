"""Order of torch's stream against the engine's own in the autograd bridge:
the engine's stream does not wait for torch's, so whatever torch still has
queued on a buffer that is handed over ends first.  Recorded calls on the CPU
(a real pair of streams would show a missing wait only now and then)."""
import types

import numpy as np
import pytest
import torch

from sre import autograd


class Calls(list):
    def note(self, what, result=None):
        self.append(what)
        return result


class Device:
    """A tensor on the GPU: conversions queue work on torch's stream, reading
    the values on the host waits for it."""

    def __init__(self, calls, name, value):
        self.calls, self.name, self.value = calls, name, value

    def detach(self):
        return self

    def double(self):
        return self.calls.note("queued " + self.name, self)

    contiguous = double

    def cpu(self):
        return self.calls.note("waited", torch.from_numpy(self.value))


def engine(calls):
    e = types.SimpleNamespace(n_types=1, n_atoms=3, n_replicas=1)
    e.set_pair_params = lambda *a: calls.note("params")
    e.compute = lambda **k: calls.note("compute")
    e.forces_to_device = lambda F: calls.note("engine writes F")
    e.stats = lambda: np.zeros((1, 4))

    def adjoint(dLdE=None, dLdF=None, tail=False, n_rc=None):
        calls.note("engine reads gF")
        return np.zeros((1, 1)), np.zeros((1, 1)), None
    e.adjoint = adjoint
    return e


@pytest.fixture
def recorded(monkeypatch):
    """sre.autograd with a torch that allocates nothing on a GPU."""
    calls = Calls()
    stream = types.SimpleNamespace(query=lambda: False,
                                   synchronize=lambda: calls.note("waited"))
    fake = types.SimpleNamespace(
        float64=torch.float64, stack=torch.stack,
        empty=lambda *a, **k: calls.note("F allocated", object()),
        from_numpy=lambda a: types.SimpleNamespace(
            to=lambda d: torch.from_numpy(a).to(d) if d != "cuda" else torch.from_numpy(a)),
        cuda=types.SimpleNamespace(current_stream=lambda *a: stream))
    monkeypatch.setattr(autograd, "torch", fake)
    return calls


def test_forward_waits_before_the_engine_writes_torchs_memory(recorded):
    one = torch.ones((1, 1), dtype=torch.float64)
    ctx = types.SimpleNamespace()
    autograd.LJEnergyForces.forward(ctx, one, one, None, engine(recorded), False)
    k = recorded.index("engine writes F")
    assert "waited" in recorded[recorded.index("F allocated"):k]


@pytest.mark.parametrize("with_energy", [True, False])
def test_backward_waits_for_the_gradient_of_the_forces(recorded, with_energy):
    f64 = torch.float64
    ctx = types.SimpleNamespace(engine=engine(recorded), tail=False, n_rc=0, rc_given=False,
                                shapes=((1, 1), (1, 1)), dtypes=(f64, f64, None))
    gE = Device(recorded, "gE", np.ones(1)) if with_energy else None
    gF = Device(recorded, "gF", np.ones((3, 3)))
    autograd.LJEnergyForces.backward(ctx, gE, gF)
    last = max(i for i, c in enumerate(recorded) if c == "queued gF")
    assert "waited" in recorded[last:recorded.index("engine reads gF")]
