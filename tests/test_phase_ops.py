"""Diagonal gates as phases in the tile passes: planner and index rules on the CPU, kernels on the GPU.

A product of G unitary gates in complex128 is within 8 * G * 2^-53 of the exact one per amplitude of a
normalised state (each gate rounds a few times); complex64 with 2^-24.
"""

import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle.cpu_sim import OracleSimulator
from projectq_amd import commands

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "native", "_build", "libphase_emu.so")


def _circuit(n, kind, seed):
    """QFT-like, random diagonal-heavy, or diagonal-only circuits of 1-qubit gates with controls."""
    rng = np.random.default_rng(seed)
    h = np.array([[1, 1], [1, -1]], dtype=complex) / np.sqrt(2.0)
    x = np.array([[0, 1], [1, 0]], dtype=complex)
    phase = lambda a: np.diag([1.0, np.exp(1j * a)])
    rz = lambda a: np.diag([np.exp(-0.5j * a), np.exp(0.5j * a)])
    out = []
    if kind == "qft":
        for q in reversed(range(n)):
            out.append((h, [q], []))
            out += [(phase(np.pi / 2 ** (q - j)), [q], [j]) for j in range(q)]
        return out
    for _ in range(12 * n):
        picks = [int(q) for q in rng.permutation(n)]
        a, c = rng.uniform(0, 2 * np.pi), int(rng.integers(0, min(n, 6)))
        pool = [(rz(a), c), (phase(a), c), (phase(np.pi), c), (np.diag([1j, 1j]), c)]
        if kind == "mixed":
            pool += [(h, 0), (x, min(c, 2)), (h, min(c, 1))]
        m, c = pool[int(rng.integers(0, len(pool)))]
        out.append((np.asarray(m, dtype=complex), picks[:1], sorted(picks[1 : 1 + c])))
    return out


def _state(n, seed):
    rng = np.random.default_rng(seed)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    return psi / np.linalg.norm(psi)


def _oracle(n, gates, psi):
    sim = OracleSimulator(1)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction(psi, list(range(n)))
    for m, t, c in gates:
        sim.apply_controlled_gate(m, t, c)
        sim.run()
    return np.array(sim.cheat_numpy()[1])


@pytest.fixture(scope="module")
def emu():
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    csrc = os.path.join(ROOT, "projectq_amd", "csrc")
    srcs = [os.path.join(ROOT, "tests", "native", "phase_emu.cpp"), os.path.join(csrc, "planner.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", csrc, *srcs, "-o", LIB], check=True)
    lib = ctypes.CDLL(LIB)
    lib.phase_error.restype = ctypes.c_char_p
    return lib


@pytest.mark.parametrize("relabel", [0, 1])
@pytest.mark.parametrize("kind", ["qft", "mixed", "diagonal"])
@pytest.mark.parametrize("n,t,lmin", [(4, 4, 2), (7, 5, 2), (9, 6, 3), (11, 8, 3)])
def test_planned_phases_equal_the_gates(emu, n, t, lmin, kind, relabel):
    gates = _circuit(n, kind, n)
    psi = _state(n, 5)
    k = np.ones(len(gates), dtype=np.uint32)
    tpos = np.array([t_[0] for _, t_, _ in gates], dtype=np.uint32)
    cmask = np.array([sum(1 << c for c in cs) for _, _, cs in gates], dtype=np.uint64)
    mats = np.concatenate([np.asarray(m, dtype=np.complex128).reshape(-1) for m, _, _ in gates])
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    passes = {}
    for phases in (0, 1):
        got, ops = psi.copy(), ctypes.c_int()
        passes[phases] = emu.phase_run(n, t, lmin, relabel, phases, len(gates), ptr(k), ptr(tpos), ptr(cmask), ptr(mats),
                                       ptr(got), ctypes.byref(ops))
        assert passes[phases] > 0, emu.phase_error()
        assert (ops.value > 0) == bool(phases)
        assert np.max(np.abs(got - _oracle(n, gates, psi))) <= 8 * len(gates) * 2.0 ** -53
    if kind == "diagonal":  # a phase fits every tile
        assert passes[1] <= passes[0]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["fusion", "window"])
@pytest.mark.parametrize("kind", ["qft", "mixed", "diagonal"])
@pytest.mark.parametrize("n,precision", [(19, "c128"), (20, "c128"), (20, "c64"), (21, "c64")])
def test_kernels_run_phases(n, precision, kind, mode):
    """19 qubits complex128 has tiles of 2^11 amplitudes, 20 qubits the full ones of both precisions."""
    from projectq_amd import Simulator

    gates = _circuit(n, kind, n)
    psi = _state(n, 6)
    kw = dict(fusion="window", planner="learned") if mode == "window" else {}
    sim = Simulator(1, precision=precision, capacity_qubits=n, **kw)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction(psi, list(range(n)))
    commands.execute(sim, [("gate", m, tuple(t), tuple(c)) for m, t, c in gates], gate_fusion=True)
    sim.run()
    eps = 2.0 ** -24 if precision == "c64" else 2.0 ** -53
    # rounding is relative to an amplitude, the largest about 5 times 2^(-n/2)
    assert np.max(np.abs(np.array(sim.cheat_numpy()[1]) - _oracle(n, gates, psi))) <= 8 * len(gates) * eps * 5 * 2.0 ** (-n / 2)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["qft", "diagonal"])
@pytest.mark.parametrize("lmin", [4, 5])
def test_kernel_of_512_threads_runs_phases(lmin, kind):
    """complex64 tiles of 2^13 amplitudes, which take 21 qubits: the tolerance as above."""
    from projectq_amd import Simulator

    n = 21
    gates = _circuit(n, kind, n + lmin)
    psi = _state(n, 7)
    sim = Simulator(1, precision="c64", capacity_qubits=n, fusion="window", planner="tile")
    sim.set_tile_params(13, 4, lmin)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction(psi, list(range(n)))
    commands.execute(sim, [("gate", m, tuple(t), tuple(c)) for m, t, c in gates], gate_fusion=True)
    sim.run()
    assert sim.last_plan()["tile_bits"] == 13
    assert np.max(np.abs(np.array(sim.cheat_numpy()[1]) - _oracle(n, gates, psi))) <= 8 * len(gates) * 2.0 ** -24 * 5 * 2.0 ** (-n / 2)
