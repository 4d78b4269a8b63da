"""Quantum circuits (quantumflow/circuits.py:35-372).

``Circuit.run`` applies its elements in order to a state (circuits.py:87-99).
For plain Gates on a state of at least ``FUSED_MIN_QUBITS`` qubits it hands
the whole gate list to the fused executor (quantumflow_amd.executor), which
plans LDS-tiled passes and fused dense blocks and runs them on the GPU;
on smaller states, runs of gates go to the gate-list kernel, many a launch;
``run(ket, fused=False)`` forces the plain path, one kernel per gate.
"""

from collections import defaultdict
from itertools import chain
from math import pi
from typing import Dict, Iterable, Iterator, Sequence, Type

from . import backend as bk
from . import config
from .channels import Density, evolve_by, evolve_kinds
from .gates import control_gate, identity_gate
from .ops import Gate, Operation
from .qubits import Qubit, Qubits
from .states import State, zero_state
from .stdgates import CCNOT, CNOT, CPHASE, H, SWAP, T, TY, TZ, X

__all__ = ['Circuit', 'count_operations', 'map_gate', 'qft_circuit',
           'reversal_circuit', 'control_circuit', 'ccnot_circuit', 'zyz_circuit',
           'phase_estimation_circuit', 'addition_circuit', 'ghz_circuit']

FUSED_MIN_QUBITS = 14


def _listed(elem, method):
    """The gate's kernel class if ``elem`` is a Gate whose ``method`` is
    Gate's own and the gate-list kernel takes it, else None."""
    if not isinstance(elem, Gate) or getattr(type(elem), method) is not getattr(Gate, method):
        return None
    if elem._host is None and elem.qubit_nb > 3:
        return None                             # stays on the device
    kind = elem.kind
    return kind if kind.listable else None


def _runs(elements, item):
    """Split ``elements`` into maximal runs for the gate-list kernel: yields
    lists of (elem, item(elem)) pairs.  An element without an item is a list of
    its own."""
    run = []
    for elem in elements:
        it = item(elem)
        if it is not None:
            run.append((elem, it))
            continue
        if run:
            yield run
            run = []
        yield [(elem, None)]
    if run:
        yield run


def _evolve_run(run, rho):
    """A density evolved by (element, kinds of evolve_kinds) pairs: each
    element's kernel gates act on its qubits' row axes, their column axes or
    both."""
    if len(run) < 2:
        for elem, gates in run:
            rho = evolve_by(gates, elem.qubits, rho)
        return rho
    n = rho.qubit_nb
    bit_of = _bits_of(rho.qubits, 2 * n)
    kinds, bits = [], []
    for elem, gates in run:
        rows = _lookup(bit_of, elem.qubits)
        cols = [b - n for b in rows]
        for kind, where in gates:
            kinds.append(kind)
            bits += rows + cols if where == 'both' else (rows if where == 'rows' else cols)
    return Density(bk.apply_gates(rho.tensor, kinds, bits), rho.qubits, rho._memory)


def _bits_of(qubits, axes):
    """Index bit of each qubit label's first axis in a tensor of ``axes`` axes:
    a state has one axis per label, a density or a gate its row axes, then its
    column axes."""
    return {q: axes - 1 - i for i, q in enumerate(qubits)}


def _lookup(bit_of, qubits):
    try:
        return [bit_of[q] for q in qubits]
    except KeyError as e:
        raise ValueError('qubit %r is not in the state' % (e.args[0],)) from None


class Circuit(Operation):
    """A sequence of operations (circuits.py:35-136)."""

    def __init__(self, elements: Iterable[Operation] = None) -> None:
        self.elements = list(elements) if elements is not None else []

    def add(self, other: 'Circuit') -> 'Circuit':
        return Circuit(self.elements + other.elements)

    def extend(self, other: Operation) -> None:
        if isinstance(other, Circuit):
            self.elements.extend(other.elements)
        else:
            self.elements.extend([other])

    def __add__(self, other: 'Circuit') -> 'Circuit':
        return self.add(other)

    def __iadd__(self, other: Operation) -> 'Circuit':
        self.extend(other)
        return self

    def __iter__(self) -> Iterator[Operation]:
        return self.elements.__iter__()

    def size(self) -> int:
        return len(self.elements)

    @property
    def qubits(self) -> Qubits:
        """Sorted unique qubits; TypeError if unsortable (circuits.py:75-85)."""
        qbs = [q for elem in self.elements for q in elem.qubits]
        qbs = list(set(qbs))
        qbs = sorted(qbs)
        return tuple(qbs)

    def flat_elements(self) -> list:
        """All elements in order with nested circuits flattened."""
        out = []
        for elem in self.elements:
            if isinstance(elem, Circuit):
                out.extend(elem.flat_elements())
            else:
                out.append(elem)
        return out

    def flat_gates(self):
        """All elements as plain Gates in order, or None if any element is
        not a Gate (nested circuits are flattened)."""
        out = self.flat_elements()
        if any(not isinstance(elem, Gate) for elem in out):
            return None
        return out

    def evolve(self, rho=None):
        """Apply every element to a Density in order (circuits.py:102-109);
        default |0...0><0...0| on the circuit's qubits."""
        if rho is None:
            rho = zero_state(qubits=self.qubits).asdensity()
        if len(self.elements) == 1:
            return self.elements[0].evolve(rho)
        run = []
        for elem in self.elements:
            how = evolve_kinds(elem)
            if callable(how):
                rho = how(_evolve_run(run, rho))
                run = []
            else:
                run.append((elem, how))
        return _evolve_run(run, rho)

    def run(self, ket: State = None, fused: bool = None) -> State:
        """Apply the circuit to ``ket`` (default |0...0> on the sorted
        qubits).  ``fused=None`` picks the fused executor for circuits on
        >= FUSED_MIN_QUBITS qubits when QUANTUMFLOW_FUSION is on: each
        maximal run of plain gates between other operations (measurements,
        resets, classical control) goes through it; the others run one by
        one in order."""
        if ket is None:
            ket = zero_state(qubits=self.qubits)
        if fused is None:
            if len(self.elements) == 1:
                return self.elements[0].run(ket)
            if config.FUSION and 0 < ket.qubit_nb < FUSED_MIN_QUBITS:
                return self._run_small(ket)
            fused = config.FUSION and ket.qubit_nb >= FUSED_MIN_QUBITS
        if not fused:
            for elem in self.elements:
                ket = elem.run(ket)
            return ket
        from .executor import run_gates
        segment = []
        for elem in self.flat_elements() + [None]:
            if isinstance(elem, Gate):
                segment.append(elem)
                continue
            if len(segment) > 1:
                ket = run_gates(segment, ket)
            elif segment:
                ket = segment[0].run(ket)
            segment = []
            if elem is not None:
                ket = elem.run(ket)
        return ket

    def _run_small(self, ket: State) -> State:
        """Runs of gates through the gate-list kernel, other elements one by
        one in order."""
        def flat(circ):
            for elem in circ.elements:
                if isinstance(elem, Circuit) and type(elem).run is Circuit.run:
                    yield from flat(elem)
                else:
                    yield elem
        for run in _runs(flat(self), lambda e: _listed(e, 'run')):
            if len(run) == 1:
                ket = run[0][0].run(ket)
                continue
            # a density's gates act on its row axes, as Gate.run's do
            bit_of = _bits_of(ket.qubits, bk.rank(ket.tensor))
            bits = [b for gate, _ in run for b in _lookup(bit_of, gate.qubits)]
            tensor = bk.apply_gates(ket.tensor, [kind for _, kind in run], bits)
            ket = State(tensor, ket.qubits, ket.memory)
        return ket

    def asgate(self) -> Gate:
        """The circuit's unitary, composed on the GPU (circuits.py:111-118):
        its gates act on the row axes of the identity."""
        qubits = self.qubits
        gate = None

        def item(elem):
            # nested circuits, among others, have no __matmul__
            if getattr(type(elem), '__matmul__', None) is Gate.__matmul__:
                return _listed(elem, 'asgate')
            return None
        for run in _runs(self.elements, item):
            if len(run) == 1:
                gate = run[0][0].asgate() @ (identity_gate(qubits) if gate is None else gate)
                continue
            n = len(qubits)
            bit_of = _bits_of(qubits, 2 * n)
            bits = [b for g, _ in run for b in _lookup(bit_of, g.qubits)]
            tensor = bk.identity_tensor(n) if gate is None else gate.tensor
            gate = Gate(tensor=bk.apply_gates(tensor, [kind for _, kind in run], bits),
                        qubits=qubits)
        return identity_gate(qubits) if gate is None else gate

    def aschannel(self):
        """The circuit's superoperator: the identity channel on its qubits
        composed with each element's channel in order (circuits.py:122-127);
        each composition is one gate-kernel pass over the superoperator."""
        chan = identity_gate(self.qubits).aschannel()
        for elem in self.elements:
            chan = elem.aschannel() @ chan
        return chan

    @property
    def H(self) -> 'Circuit':
        return Circuit([elem.H for elem in self.elements[::-1]])

    def __str__(self) -> str:
        return '\n'.join([str(elem) for elem in self.elements])


def count_operations(elements: Iterable[Operation]) -> Dict[Type[Operation], int]:
    """Count operations by type (circuits.py:139-149)."""
    op_count: Dict[Type[Operation], int] = defaultdict(int)
    for elem in elements:
        op_count[type(elem)] += 1
    return dict(op_count)


def map_gate(gate: Gate, args: Sequence[Qubits]) -> Circuit:
    """The same gate on each qubit tuple (circuits.py:152-167)."""
    circ = Circuit()
    for qubits in args:
        circ += gate.relabel(qubits)
    return circ


def qft_circuit(qubits: Qubits) -> Circuit:
    """Quantum Fourier transform (circuits.py:170-185)."""
    N = len(qubits)
    circ = Circuit()
    for n0 in range(N):
        q0 = qubits[n0]
        circ += H(q0)
        for n1 in range(n0 + 1, N):
            circ += CPHASE(pi / 2 ** (n1 - n0), qubits[n1], q0)
    circ.extend(reversal_circuit(qubits))
    return circ


def reversal_circuit(qubits: Qubits) -> Circuit:
    """Reverse the qubit order with SWAPs (circuits.py:188-194)."""
    N = len(qubits)
    circ = Circuit()
    for n in range(N // 2):
        circ += SWAP(qubits[n], qubits[N - 1 - n])
    return circ


def control_circuit(controls: Qubits, gate: Gate) -> Circuit:
    """Multi-controlled gate, Barenco et al. 1995 sec. 7.2 (circuits.py:197-225)."""
    circ = Circuit()
    if len(controls) == 1:
        q0 = controls[0]
        if isinstance(gate, X):
            circ += CNOT(q0, gate.qubits[0])
        else:
            circ += control_gate(q0, gate)
    else:
        circ += control_circuit(controls[-1:], gate ** 0.5)
        circ += control_circuit(controls[0:-1], X(controls[-1]))
        circ += control_circuit(controls[-1:], gate ** -0.5)
        circ += control_circuit(controls[0:-1], X(controls[-1]))
        circ += control_circuit(controls[0:-1], gate ** 0.5)
    return circ


def ccnot_circuit(qubits: Qubits) -> Circuit:
    """Toffoli from CNOT, H and T (Nielsen & Chuang; circuits.py:228-259)."""
    if len(qubits) != 3:
        raise ValueError('Expected 3 qubits')
    q0, q1, q2 = qubits
    circ = Circuit()
    for g in [H(q2), CNOT(q1, q2), T(q2).H, CNOT(q0, q2), T(q2), CNOT(q1, q2),
              T(q2).H, CNOT(q0, q2), T(q1), T(q2), H(q2), CNOT(q0, q1), T(q0),
              T(q1).H, CNOT(q0, q1)]:
        circ += g
    return circ


def zyz_circuit(t0: float, t1: float, t2: float, q0: Qubit) -> Circuit:
    """TZ(t0), TY(t1), TZ(t2) (circuits.py:262-268)."""
    circ = Circuit()
    circ += TZ(t0, q0)
    circ += TY(t1, q0)
    circ += TZ(t2, q0)
    return circ


def phase_estimation_circuit(gate: Gate, outputs: Qubits) -> Circuit:
    """Quantum phase estimation (circuits.py:271-303)."""
    circ = Circuit()
    circ += map_gate(H(), list(zip(outputs)))
    for cq in reversed(outputs):
        circ += control_gate(cq, gate)
        gate = gate @ gate
    circ += qft_circuit(outputs).H
    return circ


def addition_circuit(addend0: Qubits, addend1: Qubits, carry: Qubits) -> Circuit:
    """Cuccaro ripple-carry adder; result in addend1 (circuits.py:306-356)."""
    if len(addend0) != len(addend1):
        raise ValueError('Number of addend qubits must be equal')
    if len(carry) != 2:
        raise ValueError('Expected 2 carry qubits')

    def _maj(qubits: Qubits) -> Circuit:
        q0, q1, q2 = qubits
        return Circuit([CNOT(q2, q1), CNOT(q2, q0), CCNOT(q0, q1, q2)])

    def _uma(qubits: Qubits) -> Circuit:
        q0, q1, q2 = qubits
        return Circuit([CCNOT(q0, q1, q2), CNOT(q2, q0), CNOT(q0, q1)])

    qubits = [carry[0]] + list(chain.from_iterable(
        zip(reversed(addend1), reversed(addend0)))) + [carry[1]]
    circ = Circuit()
    for n in range(0, len(qubits) - 3, 2):
        circ += _maj(qubits[n:n + 3])
    circ += CNOT(qubits[-2], qubits[-1])
    for n in reversed(range(0, len(qubits) - 3, 2)):
        circ += _uma(qubits[n:n + 3])
    return circ


def ghz_circuit(qubits: Qubits) -> Circuit:
    """H then a CNOT ladder (circuits.py:359-371)."""
    circ = Circuit()
    circ += H(qubits[0])
    for q0 in range(0, len(qubits) - 1):
        circ += CNOT(qubits[q0], qubits[q0 + 1])
    return circ
