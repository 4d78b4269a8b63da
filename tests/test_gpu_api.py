"""GPU runs of the QuantumFlow API (Gate.run, Circuit.run, State, Gate @ Gate,
Circuit.asgate, DAGCircuit) on the reference's known-answer circuits and on
the seeded benchmark circuits, compared with the oracle."""
import numpy as np
import pytest
from math import pi

from oracle import qf_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qf():
    import quantumflow_amd as qf
    assert qf.backend.gpu_available()
    return qf


def build(qf, desc):
    from quantumflow_amd.workloads import build_gates
    return build_gates(desc)


def test_bits_kat(qf):
    # tests/test_gates.py:59-77
    for q in range(4):
        ket = qf.X(q).run(qf.zero_state(4))
        idx = [0, 0, 0, 0]
        idx[q] = 1
        assert ket.vec.asarray()[tuple(idx)] == 1.0
    ket = qf.zero_state(8)
    for q in (2, 4, 6):
        ket = qf.X(q).run(ket)
    assert ket.vec.asarray()[0, 0, 1, 0, 1, 0, 1, 0] == 1.0


def test_state_labels_kat(qf):
    # tests/test_states.py:54-66
    ket = qf.zero_state(range(3, -1, -1))
    ket = qf.X(0).run(ket)
    ket = qf.X(1).run(ket)
    assert ket.vec.asarray()[0, 0, 1, 1] == 1.0
    ket = ket.relabel([0, 1, 3, 4])
    assert ket.vec.asarray()[0, 0, 1, 1] == 1.0
    ket = ket.permute([4, 3, 0, 1])
    assert ket.vec.asarray()[1, 1, 0, 0] == 1.0


def test_expectation_kats(qf):
    ket = qf.H(0).run(qf.zero_state(1))
    assert abs(qf.asarray(ket.expectation([0.4, 0.6])) - 0.5) < 1e-15
    m = np.zeros([2] * 4)
    m[0, 0, 0, 0], m[1, 0, 0, 0], m[0, 1, 0, 0], m[0, 0, 1, 0], m[0, 0, 0, 1] = 42, 1, 2, 3, 4
    assert qf.asarray(qf.zero_state(4).expectation(m)) == 42
    assert abs(qf.asarray(qf.w_state(4).expectation(m)) - 2.5) < 1e-15


def test_qvm_wavefunction_kat(qf):
    # tests/test_circuits.py:43-60
    true = np.array([0.00167784 + 1.00210180e-05j, 0.50000000 - 4.99997185e-01j,
                     0.50000000 - 4.99997185e-01j, 0.00167784 + 1.00210180e-05j])
    c = qf.Circuit([qf.RY(pi / 2, 0), qf.RX(pi, 0), qf.RY(pi / 2, 1), qf.RX(pi, 1),
                    qf.CNOT(0, 1), qf.RX(-pi / 2, 1), qf.RY(4.71572463191, 1),
                    qf.RX(pi / 2, 1), qf.CNOT(0, 1), qf.RX(-2 * 2.74973750579, 0),
                    qf.RX(-2 * 2.74973750579, 1)])
    ket = c.run(qf.zero_state(2))
    assert qf.states_close(ket, qf.State(true.reshape(2, 2)))
    dag = qf.DAGCircuit(c)
    ket2 = dag.H.run(dag.run(qf.zero_state(2)))
    assert qf.states_close(ket2, qf.zero_state(2))


def test_qft_kat(qf):
    c = qf.Circuit([qf.X(2)])
    c.extend(qf.qft_circuit([0, 1, 2]))
    ket = c.run(qf.zero_state(3))
    true = np.array([0.35355339 + 0.j, 0.25 + 0.25j, 0.35355339j, -0.25 + 0.25j,
                     -0.35355339 + 0.j, -0.25 - 0.25j, -0.35355339j, 0.25 - 0.25j])
    assert np.max(np.abs(ket.vec.asarray().reshape(-1) - true)) < 1e-8


def test_adder_exact(qf):
    # tests/test_circuits.py:298-350: exact basis-state arithmetic
    circ = qf.addition_circuit([0, 1, 2], [3, 4, 5], [6, 7])
    for c0 in range(2):
        for a0 in range(8):
            for a1 in range(8):
                bits = [int(b) for b in format(a0, '03b')] + \
                       [int(b) for b in format(a1, '03b')] + [c0, 0]
                st = np.zeros([2] * 8)
                st[tuple(bits)] = 1
                out = circ.run(qf.State(st), fused=False).vec.asarray().reshape(-1)
                nz = np.nonzero(out)[0]
                assert len(nz) == 1 and out[nz[0]] == 1.0
                ob = [(nz[0] >> (7 - q)) & 1 for q in range(8)]
                assert int(''.join(str(ob[q]) for q in [7, 3, 4, 5]), 2) == a0 + a1 + c0


def test_gate_composition_on_gpu(qf):
    # ops.py:187-198 / circuits.py:111-118: asgate == product of matrices
    g = qf.zyz_circuit(0.1, 2.2, 0.5, 0).asgate()
    assert qf.gates_close(g, qf.ZYZ(0.1, 2.2, 0.5))
    c = qf.Circuit([qf.H(0), qf.CNOT(0, 1), qf.RX(0.3, 2), qf.CCNOT(2, 0, 1), qf.ISWAP(1, 2)])
    u = c.asgate()
    ref = O.circuit_unitary([(g_.matrix, g_.qubits) for g_ in c], (0, 1, 2))
    assert np.max(np.abs(u.matrix - ref)) < 1e-13


def test_layered_rotation_12q(qf):
    from quantumflow_amd.workloads import layered_rotation_circuit
    desc = layered_rotation_circuit(12, 20, seed=1)
    ref = O.run_circuit(desc, qubits=tuple(range(12)))
    for fused in (False, True):
        ket = qf.Circuit(build(qf, desc)).run(qf.zero_state(12), fused=fused)
        got = ket.vec.asarray()
        assert np.max(np.abs(got - ref)) <= 1e-12, fused
        z = qf.asarray(ket.expectation_z())
        assert np.max(np.abs(z - O.expectation_z(ref))) <= 1e-12


@pytest.mark.parametrize("fused", [False, True])
def test_mixed_circuit_20q(qf, fused):
    from quantumflow_amd.workloads import random_mixed_circuit
    n = 20
    desc = random_mixed_circuit(n, 12, seed=3)
    ref = O.run_circuit(desc, qubits=tuple(range(n)))
    ket = qf.Circuit(build(qf, desc)).run(qf.zero_state(n), fused=fused)
    got = ket.vec.asarray()
    assert np.max(np.abs(got - ref)) <= 1e-12


def test_fused_plan_reused(qf):
    """Running the same gate objects again reuses their fused plan; other
    gates get their own; every run matches the oracle."""
    from quantumflow_amd import fusion
    from quantumflow_amd.workloads import random_mixed_circuit
    n = 14
    qubits = tuple(range(n))
    desc = random_mixed_circuit(n, 10, seed=5)
    gates = build(qf, desc)
    p1 = fusion.plan_for(gates, qubits)
    assert fusion.plan_for(list(gates), qubits) is p1
    circ = qf.Circuit(gates)
    a1 = circ.run(qf.zero_state(n), fused=True).vec.asarray()
    a2 = circ.run(qf.zero_state(n), fused=True).vec.asarray()
    assert np.array_equal(a1, a2)
    assert np.max(np.abs(a1 - O.run_circuit(desc, qubits=qubits))) <= 1e-12
    desc2 = random_mixed_circuit(n, 10, seed=6)
    gates2 = build(qf, desc2)
    assert fusion.plan_for(gates2, qubits) is not p1
    a3 = qf.Circuit(gates2).run(qf.zero_state(n), fused=True).vec.asarray()
    assert np.max(np.abs(a3 - O.run_circuit(desc2, qubits=qubits))) <= 1e-12


@pytest.fixture(scope="module")
def mixed20():
    """The 28-qubit benchmark generator at 20 qubits (depth 40, seed 2024)
    and the oracle's final state."""
    from quantumflow_amd.workloads import random_mixed_circuit
    desc = random_mixed_circuit(20, 40, seed=2024)
    return desc, O.run_circuit(desc, qubits=tuple(range(20)))


@pytest.mark.parametrize("mode,width", [('unfused', 0), ('reg', 1), ('lds', 3), ('mfma', 3),
                                        ('mfma', 4), ('mfma', 5)])
def test_benchmark_circuit_20q(qf, mixed20, mode, width):
    """Amplitude error of every executor on the benchmark circuit at 20
    qubits against numpy (<= 1e-12)."""
    from quantumflow_amd.fusion import TilePlan
    from quantumflow_amd.workloads import build_gates
    desc, ref = mixed20
    gates = build_gates(desc)
    if mode == 'unfused':
        got = qf.Circuit(gates).run(qf.zero_state(20), fused=False).vec.asarray()
    else:
        plan = TilePlan(gates, tuple(range(20)), tile_bits=12, low_bits=3, block=256,
                        fuse_width=width, mode=mode)
        got = plan.run(qf.zero_state(20)).vec.asarray()
    err = float(np.max(np.abs(got - ref)))
    print("20q benchmark circuit: %d gates, mode %s width %d, max |d amp| %.3g"
          % (len(gates), mode, width, err), flush=True)
    assert err <= 1e-12


@pytest.mark.parametrize("reg_in,reg_io", [(False, False), (True, False), (False, True),
                                            (True, True)])
def test_benchmark_circuit_20q_register_io(qf, mixed20, reg_in, reg_io):
    """Passes whose first register phase loads straight from HBM and/or
    whose last stores straight to HBM against the oracle (<= 1e-12) and,
    bit for bit, against the plan that moves every tile through LDS (the
    same arithmetic in the same order)."""
    from quantumflow_amd import fusion
    from quantumflow_amd.fusion import TilePlan
    from quantumflow_amd.workloads import build_gates
    desc, ref = mixed20
    gates = build_gates(desc)
    kw = dict(tile_bits=12, low_bits=3, block=256, fuse_width=1, mode='reg')
    plan = TilePlan(gates, tuple(range(20)), reg_in=reg_in, reg_io=reg_io, **kw)
    flags = [p[1][4] for p in plan.passes if p[0] == 'tile']
    n_in = sum(bool(f & fusion.TILE_REG_IN) for f in flags)
    n_io = sum(bool(f & fusion.TILE_REG_IO) for f in flags)
    assert (n_in > 0) == reg_in and (n_io > 0) == reg_io
    got = plan.run(qf.zero_state(20)).vec.asarray()
    base = TilePlan(gates, tuple(range(20)), reg_in=False, reg_io=False, **kw)
    want = base.run(qf.zero_state(20)).vec.asarray()
    err = float(np.max(np.abs(got - ref)))
    print("20q register I/O passes: in %d, out %d of %d, max |d amp| %.3g"
          % (n_in, n_io, len(flags), err), flush=True)
    assert err <= 1e-12
    assert np.array_equal(got, want)


def test_w16_kat(qf):
    # examples/state_prep_w16.py via tests/test_examples.py:29-32
    from tests.test_oracle import w16_gates
    gates = []
    for g in w16_gates():
        if len(g) == 2:
            gates.append(qf.Gate(g[0], g[1]))
        else:
            gates.append(qf.STDGATES[g[0]](*g[1], *g[2]))
    ket = qf.Circuit(gates).run(qf.zero_state(16))
    assert qf.states_close(ket, qf.w_state(16))


@pytest.mark.parametrize("n,seed,most", [(20, 1, 300), (22, 1, 464), (23, 1, 644)])
def test_register_phase_passes_three_to_a_cu(qf, n, seed, most):
    """Passes of register phases alone in the kernel without prefetch, with
    both ends (stores from registers and in lane order) and both sizes of its
    coefficients (up to 512, and more), against the prefetching kernel on the
    same plan: the same operations in the same order, so the same bits.  At 20
    qubits a workgroup has one tile, at 22 the tiles fill the grid once and a
    third."""
    import torch
    from quantumflow_amd import fusion
    rng = np.random.default_rng(seed)
    gates = []
    for _ in range(8 * n):
        w = 12 if rng.random() < 0.8 else n
        a, b = rng.choice(w, 2, replace=False).tolist()
        gates.append([qf.RX(rng.uniform(0, 6), a), qf.H(b), qf.CPHASE(rng.uniform(0, 6), a, b),
                      qf.CNOT(a, b), qf.TY(rng.uniform(), b), qf.SWAP(a, b),
                      qf.CPHASE(rng.uniform(0, 6), b, a)][rng.integers(0, 7)])
    plan = fusion.TilePlan(gates, tuple(range(n)), tile_bits=12, low_bits=3, block=256,
                           mode='reg')
    hit = [p for k, p in plan.passes if k == 'tile' and p[4] & fusion.TILE_PHASES]
    assert {bool(p[4] & fusion.TILE_REG_IO) for p in hit} == {False, True}
    assert max(p[6] for p in hit) == most
    psi = torch.randn(2 ** n, dtype=torch.complex128, device='cuda')
    got = plan.run_inplace(psi.clone())
    plan.passes = [(k, p[:4] + (p[4] & ~fusion.TILE_PHASES,) + p[5:]) if k == 'tile' else (k, p)
                   for k, p in plan.passes]
    assert torch.equal(got, plan.run_inplace(psi.clone()))


@pytest.mark.parametrize("cfg", [
    dict(tile_bits=12, low_bits=3, block=256, mode='reg'),
    dict(tile_bits=12, low_bits=3, block=256, mode='reg', reg_in=False),
    dict(tile_bits=12, low_bits=3, block=256, mode='reg', persistent=False),
    dict(tile_bits=9, low_bits=3, block=64, mode='lds', fuse_width=4),
    dict(tile_bits=12, low_bits=3, block=256, mode='mfma'),
])
@pytest.mark.parametrize("n", [13, 16, 22])
def test_first_pass_reads_the_given_state(qf, n, cfg):
    """A plan's run leaves the state it was given as it was and returns the bits
    of the same plan run in place on a copy, for every kernel a first pass may
    take, with SWAPs folded into its store."""
    import torch
    from quantumflow_amd import fusion
    rng = np.random.default_rng(n)
    gates = []
    for _ in range(4 * n):
        a, b = rng.choice(n, 2, replace=False).tolist()
        gates.append([qf.RX(rng.uniform(0, 6), a), qf.H(b), qf.CNOT(a, b), qf.SWAP(a, b),
                      qf.CPHASE(rng.uniform(0, 6), a, b)][rng.integers(0, 5)])
    plan = fusion.TilePlan(gates, tuple(range(n)), **cfg)
    psi = torch.randn(2 ** n, dtype=torch.complex128, device='cuda')
    before = psi.clone()
    want = plan.run_inplace(before.clone())
    got = plan.run(qf.State(psi.view([2] * n), range(n)))
    assert torch.equal(got.tensor.reshape(-1), want)
    assert torch.equal(psi, before)
