"""Measurement on the device at the edges of its kernels (one workgroup up to 4096 amplitudes, chunks
above), against the oracle: single qubits, several at once, none, with known zeros and without, and
the deallocation that follows."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 4, 8, 12, 13, 17])
def test_measurements_and_deallocation(precision, n):
    from oracle.cpu_sim import OracleSimulator
    from projectq_amd import Simulator

    rng = np.random.default_rng(n)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex64 if precision == "c64" else np.complex128).astype(np.complex128)
    sims = [OracleSimulator(n), Simulator(n, precision=precision, capacity_qubits=n)]
    order = [int(q) for q in rng.permutation(n)]
    several = order[: n // 2]
    for sim in sims:
        for q in range(n):
            sim.allocate_qubit(q)
        sim.set_wavefunction(psi, list(range(n)))
    # the outcomes come from the same draws; probabilities agree to FP64 rounding of FP32 data at worst
    tol = 1e-12 if precision == "c128" else 1e-6
    for ids in ([], [order[0]], several, *([q] for q in order)):
        outcomes = [sim.measure_qubits(ids) for sim in sims]
        assert outcomes[0] == outcomes[1]
        states = [sim.cheat_numpy()[1] for sim in sims]
        assert np.max(np.abs(states[0] - states[1])) <= tol
    for q in order:
        assert sims[1].is_classical(q, 1e-12)
        assert sims[0].get_classical_value(q, 1e-12) == sims[1].get_classical_value(q, 1e-12)
        for sim in sims:
            sim.deallocate_qubit(q)
        assert np.max(np.abs(sims[0].cheat_numpy()[1] - sims[1].cheat_numpy()[1])) <= tol


def test_unmeasured_qubit_is_not_freed():
    from projectq_amd import Simulator

    sim = Simulator(1)
    for q in range(15):
        sim.allocate_qubit(q)
    psi = np.zeros(1 << 15, dtype=np.complex128)
    psi[[0, 1 << 14]] = np.sqrt(0.5)
    sim.set_wavefunction(psi, list(range(15)))
    with pytest.raises(RuntimeError):
        sim.deallocate_qubit(14)
    sim.deallocate_qubit(3)
    assert sim.is_classical(0, -1.0) is False  # every amplitude lies above a negative tolerance


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [14, 19, 22])
def test_several_qubits_with_some_fixed(precision, n):
    """Several qubits at once, some of them measured before, on subspaces that the large kernels take (22
    qubits: chunks of more than one span), then a classical check with both answers."""
    from oracle.cpu_sim import OracleSimulator
    from projectq_amd import Simulator

    rng = np.random.default_rng(100 + n)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex64 if precision == "c64" else np.complex128).astype(np.complex128)
    sims = [OracleSimulator(n), Simulator(n, precision=precision, capacity_qubits=n)]
    for sim in sims:
        for q in range(n):
            sim.allocate_qubit(q)
        sim.set_wavefunction(psi, list(range(n)))
    assert sims[1].is_classical(n - 1, 1e-30) is False
    tol = 1e-12 if precision == "c128" else 1e-6
    for ids in ([n - 1], [0, n - 1], [5, 0, 2]):
        outcomes = [sim.measure_qubits(ids) for sim in sims]
        assert outcomes[0] == outcomes[1]
        assert np.max(np.abs(sims[0].cheat_numpy()[1] - sims[1].cheat_numpy()[1])) <= tol
        for q in range(n):
            assert sims[0].is_classical(q, 1e-30) == sims[1].is_classical(q, 1e-30)
