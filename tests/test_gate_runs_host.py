"""How circuits hand their gates to the gate-list kernel (no GPU: the calls
that would launch are recorded instead)."""
from types import SimpleNamespace

import numpy as np
import pytest

import quantumflow_amd as qf
from quantumflow_amd import circuits, ops


@pytest.fixture
def recorded(monkeypatch):
    """Stands in for the kernels: states keep their tensor, and every gate
    application is recorded as its index bits."""
    log = []

    def apply_gates(tensor, kinds, bits):
        bits = list(bits)
        for kind in kinds:
            log.append(tuple(bits[:kind.k]))
            del bits[:kind.k]
        assert not bits
        return tensor

    def tensormul(kind, tensor, indices):
        log.append(tuple(np.ndim(tensor) - 1 - i for i in indices))
        return tensor

    def state(tensor, qubits, memory):
        return SimpleNamespace(tensor=tensor, qubits=tuple(qubits), memory=memory,
                               qubit_nb=len(qubits))

    bk = SimpleNamespace(apply_gates=apply_gates, tensormul=tensormul, rank=np.ndim,
                         classify=ops.bk.classify)
    monkeypatch.setattr(circuits, 'bk', bk)
    monkeypatch.setattr(ops, 'bk', bk)
    monkeypatch.setattr(circuits, 'State', state)
    monkeypatch.setattr(ops, 'State', state)
    return SimpleNamespace(log=log, state=state)


@pytest.mark.parametrize("rank", [1, 2])
def test_run_and_plain_path_name_the_same_bits(recorded, rank):
    # rank 2: a density, whose gates act on its row axes, the first ones
    labels = ('a', 'b', 'c')
    ket = recorded.state(np.zeros([2] * (3 * rank)), labels, {})
    circ = qf.Circuit([qf.X('a'), qf.CNOT('c', 'a'), qf.RX(0.3, 'b')])
    circ.run(ket)
    got, recorded.log[:] = list(recorded.log), []
    circ.run(ket, fused=False)
    top = 3 * rank - 1
    assert recorded.log == [(top,), (top - 2, top), (top - 1,)]
    assert got == recorded.log
