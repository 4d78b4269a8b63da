"""How circuits hand their gates to the gate-list kernel (no GPU: the calls
that would launch are recorded instead)."""
import copy
import pickle
from types import SimpleNamespace

import numpy as np
import pytest

import quantumflow_amd as qf
from oracle import qf_oracle as O
from quantumflow_amd import channels, circuits, gates, ops


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


@pytest.fixture
def on_host(monkeypatch):
    """The gate kernels' results from the oracle, on host arrays."""
    def tensormul(kind, tensor, indices):
        m = kind.matrix.reshape([2] * (2 * kind.k))
        return O.tensormul(m, tensor, [int(i) for i in indices])

    def apply_gates(tensor, kinds, bits):
        bits = list(bits)
        for kind in kinds:
            axes = [np.ndim(tensor) - 1 - b for b in bits[:kind.k]]
            tensor = tensormul(kind, tensor, axes)
            del bits[:kind.k]
        return tensor

    bk = SimpleNamespace(
        apply_gates=apply_gates, tensormul=tensormul, rank=np.ndim, classify=ops.bk.classify,
        identity_tensor=lambda n: np.eye(2 ** n, dtype=complex).reshape([2] * (2 * n)),
        astensorproduct=lambda a: np.reshape(a, [2] * int(np.log2(np.size(a)))))
    for module in (circuits, gates, ops):
        monkeypatch.setattr(module, 'bk', bk, raising=False)


def test_asgate_of_nested_circuits(on_host):
    x, h, cx, rz = qf.X(1), qf.H(0), qf.CNOT(0, 1), qf.RZ(0.4, 1)
    want = cx.matrix @ np.kron(h.matrix, np.eye(2)) @ np.kron(np.eye(2), rz.matrix @ x.matrix)
    C = qf.Circuit
    for circ in (C([C([x]), rz, h, cx]), C([x, rz, C([h, cx])]), C([C([x, C([rz])]), C([h]), cx]),
                 C([C([C([x, rz, h, cx])])])):
        got = circ.asgate()
        assert got.qubits == (0, 1)
        # a product of four unitaries of two terms a row
        np.testing.assert_allclose(got.matrix, want, rtol=0, atol=16 * 2.0 ** -53)


def test_asgate_keeps_the_error_of_operations_without_a_gate(on_host):
    with pytest.raises(NotImplementedError):
        qf.Circuit([qf.X(0), qf.Measure(0)]).asgate()
    with pytest.raises(TypeError):
        qf.Circuit([qf.X(0), qf.Damping(0.1, 0)]).asgate()


@pytest.mark.parametrize("gate", [qf.RX(0.3, 0), qf.RZ(0.7, 1), qf.ISWAP(0, 1)])
def test_gates_are_copied_and_pickled_after_a_run(gate):
    # what a run leaves with the gate: its class and native record
    rec = gate.kind.record()
    assert gate.kind.record() is rec
    copies = [copy.copy(gate.kind), copy.deepcopy(gate).kind]
    copies += [pickle.loads(pickle.dumps(gate, protocol)).kind for protocol in (2, 3, 4, 5)]
    for kind in copies:
        assert (kind.kind, kind.k) == (gate.kind.kind, gate.kind.k)
        for name in ('matrix', 'diag', 'src', 'phase'):
            a, b = getattr(kind, name), getattr(gate.kind, name)
            assert (a is None and b is None) or np.array_equal(a, b)
        # a record of its own, with the same contents
        own = kind.record()
        assert own[0] != rec[0]
        assert (own[1].kind, own[1].k) == (rec[1].kind, rec[1].k)
        for a, b in zip(own[2:], rec[2:]):
            assert (a is None and b is None) or np.array_equal(a, b)


def test_class_pickled_without_a_record_slot_loads():
    kind = qf.ISWAP(0, 1).kind
    old = type(kind).__new__(type(kind))
    old.__setstate__((None, {n: getattr(kind, n) for n in kind.__slots__ if n != '_record'}))
    assert old.record()[1].k == 2


@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 5, 6])
def test_gate_classes_by_width(k):
    # read as lists up to 3 qubits, by numpy above; dense from 6 on
    rng = np.random.default_rng(k)
    dim = 2 ** k
    phases = np.exp(1j * rng.uniform(0, 6, dim))
    perm = np.roll(np.arange(dim), 1)
    zero_row = np.diag(phases)
    zero_row[0, 0] = 0
    twice = np.eye(dim)[np.zeros(dim, dtype=int)]          # one entry a row, no permutation
    moves = dim > 1
    for m, kind, src, phase in [
            (np.diag(phases), 'diagonal', None, None), (zero_row, 'diagonal', None, None),
            (np.eye(dim)[perm], 'monomial' if moves else 'diagonal', perm, None),
            (phases[:, None] * np.eye(dim)[perm], 'monomial' if moves else 'diagonal', perm, phases),
            (twice, 'dense' if moves else 'diagonal', None, None),
            (np.full((dim, dim), np.nan), 'dense' if moves else 'diagonal', None, None)]:
        got = ops.bk.classify(m)
        assert got.kind == ('dense' if k > 5 else kind)
        if got.kind == 'diagonal':
            assert np.array_equal(got.diag, np.diag(m).astype(complex), equal_nan=True)
        if got.kind == 'monomial':
            assert got.src.dtype == np.int32 and np.array_equal(got.src, src)
            assert got.phase is None if phase is None else np.array_equal(got.phase, phase)


def test_classes_of_wide_gates_cost_little_more():
    # a 5-qubit matrix has 16 times the entries of a 3-qubit one; read entry by
    # entry it took 8 times as long, by numpy twice
    import timeit
    cost = []
    for k in (3, 5):
        m = np.linalg.qr(np.random.default_rng(k).normal(size=(2 ** k, 2 ** k)))[0].astype(complex)
        cost.append(min(timeit.repeat(lambda: ops.bk.classify(m), number=200, repeat=5)))
    assert cost[1] <= 4 * cost[0]


def test_elements_between_runs_are_classified_once(monkeypatch):
    # a dense 2-qubit channel is no gate of a list, and alone between two of
    # them neither is a gate: evolving them costs what their own evolve does
    rng = np.random.default_rng(3)
    u = np.linalg.qr(rng.normal(size=(4, 4)) + 1j * rng.normal(size=(4, 4)))[0]
    chan = qf.Gate(u, [0, 1]).aschannel()
    kraus = qf.Kraus([qf.Gate(u, [0, 1]), qf.CNOT(0, 1)], [0.5, 0.5])
    rx = qf.RX(0.3, 0)
    classified, applied = [], []

    def classify(m):
        classified.append(m)
        return ops.bk.classify(m)

    def tensormul(kind, tensor, indices):
        applied.append((kind.k, tuple(indices)))
        return tensor

    def density(tensor, qubits, memory):
        return SimpleNamespace(tensor=tensor, qubits=tuple(qubits), _memory=memory,
                               qubit_nb=len(qubits))
    stub = SimpleNamespace(classify=classify, tensormul=tensormul, rank=np.ndim)
    for module in (circuits, channels):
        monkeypatch.setattr(module, 'bk', stub)
        monkeypatch.setattr(module, 'Density', density, raising=False)
    monkeypatch.setattr(channels.Kraus, '_evolve_terms', lambda self, rho: rho,
                        raising=False)
    rho = density(np.zeros([2] * 6), (0, 1, 2), {})
    for circ in (qf.Circuit([chan, rx, chan]), qf.Circuit([kraus, rx, kraus]),
                 qf.Circuit([rx]), qf.Circuit([chan])):
        del classified[:], applied[:]
        circ.evolve(rho)
        assert len(classified) == len(circ.elements)
        assert applied == [(4, (0, 1, 3, 4)) if e is chan else (2, (0, 3))
                           for e in circ.elements if e is not kraus]
