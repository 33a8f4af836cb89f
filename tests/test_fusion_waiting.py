"""Complete blocks that wait under the reference's fusion rule (GPU): what runs them, and what of the queue is
left when it does.

The reference values come from the oracle or the mathematics.  8 roundings of half an ulp per gate bound the
error: 8 * gates * 2^-24 (complex64) or 2^-53 (complex128) on amplitudes of at most 1.
"""

import numpy as np
import pytest

from oracle.cpu_sim import OracleSimulator

pytestmark = pytest.mark.gpu

EPS = {"c64": 2.0 ** -24, "c128": 2.0 ** -53}
H = np.array([[1, 1], [1, -1]], dtype=complex) / np.sqrt(2.0)
X = np.array([[0, 1], [1, 0]], dtype=complex)
SQUEEZE = np.diag([1.0, 0.5]).astype(complex)

BREAKS = {
    "allocate": lambda sim: sim.allocate_qubit(3),
    "synchronize": lambda sim: sim.synchronize(),
    "stats": lambda sim: sim.stats(),
    "reset_stats": lambda sim: sim.reset_stats(),
    "set_profiling": lambda sim: sim.set_profiling(True),
}


def _amplitudes(sim):
    return np.array(sim.cheat_numpy()[1])


@pytest.mark.parametrize("what", list(BREAKS))
def test_norm_guard_keeps_a_waiting_gate(what):
    """A gate that is not unitary waits in the open block while the block before it runs: the norm guard
    still stops at it, and the gates behind it do not scale its norm away."""
    from projectq_amd import Simulator

    sim, ref = Simulator(3, precision="c64"), OracleSimulator(3)
    for s in (sim, ref):
        for q in range(3):
            s.allocate_qubit(q)
            s.apply_controlled_gate(H, [q], [])
        s.run()
        s.apply_controlled_gate(H, [0], [])
        s.apply_controlled_gate(SQUEEZE, [2], [1])  # does not fit the block of the H: closes it, opens its own
        if s is sim or what == "allocate":
            BREAKS[what](s)
        s.run()
        for _ in range(40):  # more drift than the guard's budget
            s.apply_controlled_gate(H, [0], [])
            s.run()
    got, want = _amplitudes(sim), _amplitudes(ref)
    assert np.linalg.norm(want) < 0.95
    assert np.max(np.abs(got - want)) <= 8 * 45 * EPS["c64"]


@pytest.mark.parametrize("n,precision", [(4, "c64"), (4, "c128"), (13, "c64"), (13, "c128"), (19, "c128"), (20, "c64")])
def test_gates_without_targets(n, precision):
    """A 1x1 matrix without targets, with and without controls, inside blocks of other gates.  19 qubits
    complex128 and 20 complex64 have full tiles."""
    from projectq_amd import Simulator

    swap = np.eye(4, dtype=complex)[[0, 2, 1, 3]]
    sim, ref = Simulator(3, precision=precision, capacity_qubits=n), OracleSimulator(3)
    rng = np.random.default_rng(n)
    gates = 0
    for q in range(n):
        sim.allocate_qubit(q)
        ref.allocate_qubit(q)
    for _ in range(4):
        a, b, c, d = (int(q) for q in rng.permutation(n)[:4])
        block = [(H, [a], []), (np.array([[np.exp(0.3j)]]), [], []), (H, [b], []), (np.array([[1j]]), [], [a]),
                 (swap, [a, b], []), (H, [c], []), (X, [d], [a])]
        for s in (sim, ref):
            for m, t, k in block:
                s.apply_controlled_gate(np.asarray(m, dtype=complex), t, k)
        gates += len(block)
    sim.run()
    ref.run()
    assert np.max(np.abs(_amplitudes(sim) - _amplitudes(ref))) <= 8 * gates * EPS[precision]


@pytest.mark.parametrize("shape", ["env", (10, 4, 8), (6, 4, 5)])
@pytest.mark.parametrize("precision", ["c64", "c128"])
def test_tile_planner_settings_leave_fusion_alone(precision, shape, monkeypatch):
    """The tile planner's shape, here too narrow for three targets, has no say in what gate fusion runs."""
    from projectq_amd import Simulator

    n = 12
    rng = np.random.default_rng(7)
    q, _ = np.linalg.qr(rng.normal(size=(8, 8)) + 1j * rng.normal(size=(8, 8)))
    if shape == "env":
        monkeypatch.setenv("PROJECTQ_AMD_TILE", "6:4")
    sim, ref = Simulator(3, precision=precision), OracleSimulator(3)
    if shape != "env":
        sim.set_tile_params(*shape)
    gates = 0
    for s in (sim, ref):
        for k in range(n):
            s.allocate_qubit(k)
    for k in range(6):
        picks = [int(v) for v in np.random.default_rng(k).permutation(n)[:3]]
        for s in (sim, ref):
            s.apply_controlled_gate(np.ascontiguousarray(q), picks, [])
            s.apply_controlled_gate(H, [picks[0]], [])
        gates += 2
    sim.run()
    ref.run()
    assert np.max(np.abs(_amplitudes(sim) - _amplitudes(ref))) <= 8 * 8 * gates * EPS[precision]


@pytest.mark.parametrize("n,k,precision,blocks", [
    (12, 5, "c64", False), (12, 5, "c128", False), (21, 3, "c128", False), (21, 3, "c64", False),
    (23, 5, "c128", True), (24, 5, "c64", True),
])
def test_wide_gates_take_the_faster_way(n, k, precision, blocks):
    """Gates of 5 targets on large states run one per block (as many passes as gates), else the waiting
    blocks share passes.  A row of a gate adds 2^k products."""
    from projectq_amd import Simulator

    sim, ref = Simulator(3, precision=precision, capacity_qubits=n), OracleSimulator(3)
    rng = np.random.default_rng(n + k)
    for q in range(n):
        sim.allocate_qubit(q)
        ref.allocate_qubit(q)
    sim.run()
    sim.reset_stats()
    count = 6
    for _ in range(count):
        u, _ = np.linalg.qr(rng.normal(size=(1 << k, 1 << k)) + 1j * rng.normal(size=(1 << k, 1 << k)))
        targets = [int(q) for q in rng.permutation(n)[:k]]
        for s in (sim, ref):
            s.apply_controlled_gate(np.ascontiguousarray(u), targets, [])
    sim.run()
    ref.run()
    passes = sim.stats()["passes"]
    assert passes == count if blocks else passes < count
    assert np.max(np.abs(_amplitudes(sim) - _amplitudes(ref))) <= 8 * (1 << k) * count * EPS[precision]


@pytest.mark.parametrize("precision", ["c64", "c128"])
def test_greedy_window_with_many_controls(precision):
    """A gate of 19 controls behind others: the block it does not fit is closed without building the matrix of
    both."""
    from projectq_amd import Simulator

    n = 20
    z = np.diag([1, -1]).astype(complex)
    sim, ref = Simulator(3, precision=precision, capacity_qubits=n, fusion="window", planner="greedy"), OracleSimulator(3)
    gates = [(H, [q], []) for q in range(n)] + [(z, [0], list(range(1, n)))] + [(H, [q], []) for q in range(n)]
    for s in (sim, ref):
        for q in range(n):
            s.allocate_qubit(q)
    for m, t, c in gates:
        sim.apply_controlled_gate(m, t, c)
        ref.apply_controlled_gate(m, t, c)
        ref.run()
    sim.run()
    assert np.max(np.abs(_amplitudes(sim) - _amplitudes(ref))) <= 8 * len(gates) * EPS[precision]
