"""Runs of gates through the gate-list kernel (qfx_apply_gates): small states,
densities and composed gates against the per-gate path and the oracle."""
import numpy as np
import pytest

from oracle import qf_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qf():
    import quantumflow_amd as qf
    assert qf.backend.gpu_available()
    return qf


def _rand_state(n, rng):
    v = rng.normal(size=2 ** n) + 1j * rng.normal(size=2 ** n)
    return (v / np.linalg.norm(v)).reshape([2] * n)


def _rand_gates(qf, n, count, rng, wide=True):
    """Gates of every class and width that fits n qubits."""
    names = [('H', 0, 1), ('X', 0, 1), ('T', 0, 1), ('RX', 1, 1), ('RY', 1, 1), ('RZ', 1, 1)]
    if n > 1:
        names += [('CNOT', 0, 2), ('CZ', 0, 2), ('SWAP', 0, 2), ('ISWAP', 0, 2), ('XX', 1, 2)]
    if n > 2:
        names += [('CCNOT', 0, 3), ('CSWAP', 0, 3), ('U3', 0, 3)]
    if n > 3 and wide:
        names += [('P4', 0, 4), ('D4', 0, 4), ('U4', 0, 4)]
    out = []
    for _ in range(count):
        name, np_, k = names[rng.integers(len(names))]
        q = [int(i) for i in rng.permutation(n)[:k]]
        if name in ('U3', 'U4'):
            a = rng.normal(size=(2 ** k, 2 ** k)) + 1j * rng.normal(size=(2 ** k, 2 ** k))
            out.append(qf.Gate(np.linalg.qr(a)[0], q))
        elif name == 'P4':
            out.append(qf.Gate(np.eye(16)[rng.permutation(16)], q))
        elif name == 'D4':
            out.append(qf.Gate(np.diag(np.exp(1j * rng.uniform(0, 6, 16))), q))
        else:
            out.append(qf.STDGATES[name](*rng.uniform(0, 6, np_), *q))
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 10, 11, 12, 13])
@pytest.mark.parametrize("count", [2, 7, 150])
def test_small_circuits_match_per_gate_path(qf, n, count):
    # every block size, batches that fill the argument space, wide gates that
    # break a run
    rng = np.random.default_rng(100 * n + count)
    psi = _rand_state(n, rng)
    circ = qf.Circuit(_rand_gates(qf, n, count, rng))
    ket = qf.State(psi, range(n))
    got = circ.run(ket).vec.asarray()
    plain = circ.run(ket, fused=False).vec.asarray()
    # the same operations in the same order
    assert np.array_equal(got, plain)
    assert np.array_equal(ket.vec.asarray(), psi)


def test_small_circuit_with_measurement_and_nested_circuit(qf):
    rng = np.random.default_rng(5)
    n = 6
    inner = qf.Circuit(_rand_gates(qf, n, 5, rng))
    circ = qf.Circuit(_rand_gates(qf, n, 4, rng)) + inner
    circ += qf.Measure(2, 'c')
    circ.elements += _rand_gates(qf, n, 6, rng)
    np.random.seed(3)
    a = circ.run()
    np.random.seed(3)
    b = circ.run(fused=False)
    assert np.array_equal(a.vec.asarray(), b.vec.asarray())
    assert a.memory['c'] == b.memory['c']
    with pytest.raises(ValueError):
        qf.Circuit([qf.H(0), qf.X(7)]).run(qf.zero_state(2))


@pytest.mark.parametrize("n", [1, 2, 3, 6, 7, 8])
def test_run_on_a_density_matches_per_gate_path(qf, n):
    # run multiplies a density's rows alone; 2 to 16 index bits
    rng = np.random.default_rng(60 + n)
    circ = qf.Circuit(_rand_gates(qf, n, 25, rng))
    rho = qf.State(_rand_state(n, rng), range(n)).asdensity()
    got = circ.run(rho)
    plain = circ.run(rho, fused=False)
    assert type(got) is type(plain) and got.qubits == plain.qubits
    # 25 gates on entries of at most 1, up to 16 terms a sum: gates that share
    # no qubit may change places
    assert np.max(np.abs(got.vec.asarray() - plain.vec.asarray())) <= 25 * 16 * 2.0 ** -53


@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 7, 8])
def test_density_circuits_match_element_by_element(qf, n):
    # 2n from 2 to 16 index bits: whole-state tiles, then passes of 12 bits
    rng = np.random.default_rng(40 + n)
    circ = qf.Circuit()
    for g in _rand_gates(qf, n, 30, rng, wide=False):
        circ += g
        q = int(rng.integers(n))
        circ += [qf.Depolarizing(0.02, q), qf.Damping(0.03, q), qf.Dephasing(0.1, q)][q % 3]
    if n > 1:
        circ += qf.CNOT(0, n - 1).aschannel()
        circ += qf.Kraus([qf.CZ(0, 1), qf.CNOT(1, 0)], [0.25, 0.75])
    rho0 = qf.State(_rand_state(n, rng), range(n)).asdensity()
    got = circ.evolve(rho0)
    want = rho0
    for elem in circ.elements:
        want = elem.evolve(want)
    a, b = got.vec.asarray(), want.vec.asarray()
    # up to 80 maps on entries of at most 1: gates that share no qubit may
    # change places, a rounding of 2^-53 times their 16 terms each
    assert np.max(np.abs(a - b)) <= 80 * 16 * 2.0 ** -53
    assert abs(complex(got.trace().item()) - 1) <= 1e-12


def test_long_lists_take_linear_time(qf):
    # 16 index bits, where a list is many passes: a gate of 128000 costs what
    # one of 4000 does (about 1 us; 3.3 us when every pass read the whole list)
    import time
    import torch
    from quantumflow_amd import backend as bk
    rng = np.random.default_rng(2)
    state = bk.zero_state_tensor(16)
    rx, cnot = qf.RX(0.4, 0).kind, qf.CNOT(0, 1).kind

    def per_gate(count):
        kinds, bits = [], []
        for i in range(count):
            kinds.append(cnot if i % 3 == 2 else rx)
            bits += [int(b) for b in rng.permutation(16)[:kinds[-1].k]]
        best = np.inf
        for _ in range(3):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            bk.apply_gates(state, kinds, bits)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best / count
    short = per_gate(4000)
    assert per_gate(128000) <= 2 * short


@pytest.mark.parametrize("k", [1, 3, 6, 7, 8])
def test_composed_gate_matches_products(qf, k):
    rng = np.random.default_rng(70 + k)
    gates = _rand_gates(qf, k, 40, rng)
    gates += [qf.RX(0.1 * q, q) for q in range(k)]          # every qubit is named
    circ = qf.Circuit(gates)
    got = circ.asgate()
    want = np.eye(2 ** k, dtype=complex).reshape([2] * (2 * k))
    for g in gates:
        want = O.tensormul(g.matrix.reshape([2] * (2 * g.qubit_nb)), want, list(g.qubits))
    assert got.qubits == tuple(range(k))
    assert np.max(np.abs(got.matrix - want.reshape(2 ** k, 2 ** k))) <= 1e-13


@pytest.mark.parametrize("n", [2, 5, 8])
def test_nested_circuits_match_flat_ones(qf, n):
    rng = np.random.default_rng(90 + n)
    gates = _rand_gates(qf, n, 12, rng) + [qf.RX(0.1 * q, q) for q in range(n)]
    flat = qf.Circuit(gates)
    nested = qf.Circuit([qf.Circuit(gates[:3]), gates[3], qf.Circuit([qf.Circuit(gates[4:6])]),
                         qf.Circuit(gates[6:9])] + gates[9:])
    ket = qf.State(_rand_state(n, rng), range(n))
    assert np.array_equal(nested.run(ket).vec.asarray(), flat.run(ket).vec.asarray())
    # 20 unitaries of at most 16 terms a row, multiplied in another grouping
    assert nested.asgate().qubits == flat.asgate().qubits
    assert np.max(np.abs(nested.asgate().matrix - flat.asgate().matrix)) <= 20 * 16 * 2.0 ** -53


def test_circuits_are_copied_and_pickled_after_a_run(qf):
    import copy
    import pickle
    rng = np.random.default_rng(8)
    circ = qf.Circuit(_rand_gates(qf, 4, 12, rng))
    ket = qf.State(_rand_state(4, rng), range(4))
    want = circ.run(ket).vec.asarray()
    circ.asgate()
    for g in circ.elements:
        g.tensor                                # the device copy goes along
    for other in (copy.deepcopy(circ), pickle.loads(pickle.dumps(circ))):
        assert np.array_equal(other.run(ket).vec.asarray(), want)


def test_records_are_checked(qf):
    from quantumflow_amd import _native, backend as bk
    ket = qf.zero_state(3).tensor
    x = qf.X(0).kind
    with pytest.raises(ValueError):
        bk.apply_gates(ket, [x, x], [0, 3])                 # bit out of range
    with pytest.raises(ValueError):
        bk.apply_gates(ket, [qf.CNOT(0, 1).kind], [1, 1])   # repeated bit
    with pytest.raises(ValueError):
        bk.apply_gates(ket, [], [])
    wide = bk.classify(np.linalg.qr(np.random.default_rng(0).normal(size=(16, 16)))[0])
    assert not wide.listable
    with pytest.raises(ValueError):
        bk.apply_gates(qf.zero_state(5).tensor, [wide], [0, 1, 2, 3])
