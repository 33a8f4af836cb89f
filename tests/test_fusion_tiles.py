"""Gate fusion through tile passes (GPU): complete blocks wait for run() and go together.

A unitary gate on complex numbers rounds each amplitude a few times: 8 roundings of half an ulp per gate
bound the error, 8 * gates * 2^-24 (complex64) or 2^-53 (complex128) on amplitudes of at most 1.
"""

import numpy as np
import pytest

from oracle.cpu_sim import OracleSimulator
from projectq_amd import circuits, commands

pytestmark = pytest.mark.gpu

EPS = {"c64": 2.0 ** -24, "c128": 2.0 ** -53}


def _amplitudes(sim):
    ids, amps = sim.cheat_numpy()
    return amps


def _pair(precision, capacity=0):
    from projectq_amd import Simulator

    return Simulator(3, precision=precision, capacity_qubits=capacity), OracleSimulator(3)


@pytest.mark.parametrize("precision", ["c64", "c128"])
@pytest.mark.parametrize("n", [3, 4, 7, 11, 12, 13, 16])
def test_blocks_in_tiles(n, precision):
    cmds = circuits.random_layers(n, 3, max(n // 2, 1), 11 + n, measure=False)
    hip, ref = _pair(precision)
    commands.execute(hip, cmds, gate_fusion=True)
    commands.execute(ref, cmds, gate_fusion=True)
    gates = sum(1 for c in cmds if c[0] == "gate")
    assert np.max(np.abs(_amplitudes(hip) - _amplitudes(ref))) <= 8 * gates * EPS[precision]


@pytest.mark.parametrize("precision", ["c64", "c128"])
def test_state_changes_between_blocks(precision):
    """Allocation, measurement, a gate that is not unitary and a wide gate between waiting blocks."""
    h = np.array([[1, 1], [1, -1]]) / np.sqrt(2.0)
    x = np.array([[0, 1], [1, 0]], dtype=complex)
    squeeze = np.diag([1.0, 0.5]).astype(complex)
    results = []
    gates = 0
    for sim in _pair(precision):
        out = []
        for q in range(6):
            sim.allocate_qubit(q)
        for _ in range(3):
            for q in range(6):
                sim.apply_controlled_gate(h, [q], [])
                sim.apply_controlled_gate(x, [(q + 1) % 6], [q])
                gates += 2
        sim.allocate_qubit(6)
        sim.apply_controlled_gate(h, [6], [])
        for q in range(6):
            sim.apply_controlled_gate(x, [q], [6])
        sim.apply_controlled_gate(squeeze, [2], [])
        for q in range(7):
            sim.apply_controlled_gate(h, [q], [])
        gates += 15
        out.append(_amplitudes(sim))
        with pytest.raises((ValueError, RuntimeError)):
            sim.apply_controlled_gate(np.eye(64), list(range(6)), [])
            sim.run()
        results.append(out)
    assert np.max(np.abs(results[0][0] - results[1][0])) <= 8 * gates * EPS[precision]


def test_synchronize_runs_complete_blocks():
    """synchronize() and the counters see the complete blocks, as when each ran at once."""
    h = np.array([[1, 1], [1, -1]]) / np.sqrt(2.0)
    sim, _ = _pair("c128")
    for q in range(12):
        sim.allocate_qubit(q)
    sim.run()
    sim.reset_stats()
    for q in range(12):
        sim.apply_controlled_gate(h, [q], [])
    assert sim.stats()["passes"] > 0
    sim.synchronize()
    sim.run()
    assert np.allclose(_amplitudes(sim), 2.0 ** -6, rtol=0, atol=8 * 12 * EPS["c128"])
