"""Pauli sums applied to a state (projectq_amd/csrc/pauli_sum.hip): the plan against brute force on the
CPU; qubit operators and time evolution against the oracle at the edges of the tile shapes."""

import ctypes

import numpy as np
import pytest

from test_energy_plan import CSRC, NATIVE  # noqa: F401  (paths)


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    import os
    import subprocess

    lib = str(tmp_path_factory.mktemp("sum") / "libenergy_emu.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, os.path.join(NATIVE, "energy_emu.cpp"),
                    os.path.join(CSRC, "energy_plan.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib).sum_emu


@pytest.mark.parametrize("c64", [False, True])
@pytest.mark.parametrize("kind", ["random", "local"])
@pytest.mark.parametrize("n,count", [(1, 3), (5, 9), (8, 20), (9, 6), (11, 40), (12, 25), (13, 60)])
def test_plan_equals_brute_force(emu, c64, kind, n, count):
    rng = np.random.default_rng(n * 100 + count)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    x, z = rng.integers(0, 1 << n, size=count), rng.integers(0, 1 << n, size=count)
    if kind == "local":
        x = x & (1 << rng.integers(0, n, size=count))
    x[count // 2] = x[0]  # two strings with one x
    x[-1] = z[-1] = 0     # the identity
    c = rng.normal(size=count) + 1j * rng.normal(size=count)
    c[0], c[1] = 0.5, 2j  # real and imaginary coefficients make one string, others two
    out = np.zeros(2 << n)
    dbl, u64 = ctypes.c_double, ctypes.c_ulonglong * count
    ptr = lambda a: a.ctypes.data_as(ctypes.POINTER(dbl))  # noqa: E731
    outside = emu(ptr(psi), n, int(c64), u64(*map(int, x)), u64(*map(int, z)), ptr(c), count, ptr(out))
    assert outside >= 0 and (outside > 0 or n < 13 or kind == "local")
    i = np.arange(1 << n)
    want = np.zeros(1 << n, dtype=complex)
    for t in range(count):
        j = i ^ x[t]
        want += c[t] * (1 - 2 * np.array([bin(v).count("1") & 1 for v in j & z[t]])) * psi[j]
    assert np.max(np.abs(out.view(complex) - want)) <= 1e-15 * count * np.sum(np.abs(c))


def simulators(n, precision, seed):
    from oracle.cpu_sim import OracleSimulator
    from projectq_amd import Simulator

    rng = np.random.default_rng(seed)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex64 if precision == "c64" else np.complex128).astype(np.complex128)
    sims = (OracleSimulator(1), Simulator(1, precision=precision, capacity_qubits=n))
    for sim in sims:
        for q in range(n):
            sim.allocate_qubit(q)
        sim.set_wavefunction(psi, list(range(n)))
    return sims


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 6, 9, 12, 15])
def test_gpu_operator_and_evolution(precision, n):
    from projectq_amd import circuits

    sims = simulators(n, precision, n)
    rng = np.random.default_rng(n)
    ids = [int(q) for q in rng.permutation(n)]
    real = [t for t in circuits.random_pauli_operator(n, 14, n) if t[0]] + [([(0, "Z")], 0.3)]
    size = sum(abs(c) for _, c in real)
    # FP64: a Taylor series of a dozen terms a step; complex64 stores every term and the sum in FP32
    tol = 1e-12 if precision == "c128" else 5e-6
    runs = [(real, 0.15, ids, []), (real + [([], 0.8)], -0.4, ids, []), ([([], 1.5)], 0.3, ids, [])]
    if n > 5:
        short = [([op for op in t if op[0] < 3] or [(1, "X")], c) for t, c in real]
        runs.append((short + [([], -0.7)], 0.2, ids[:3], ids[3:5]))
    for terms, time, targets, ctrl in runs:
        for sim in sims:
            sim.emulate_time_evolution(terms, time, targets, ctrl)
        assert np.max(np.abs(sims[0].cheat_numpy()[1] - sims[1].cheat_numpy()[1])) <= tol
    complex_terms = [(t, c * (0.6 - 0.8j) / size) for t, c in real]
    for sim in sims:
        sim.apply_qubit_operator(complex_terms, ids)
    assert np.max(np.abs(sims[0].cheat_numpy()[1] - sims[1].cheat_numpy()[1])) <= tol


@pytest.mark.gpu
def test_gpu_operator_too_large_for_the_arena():
    sims = simulators(4, "c128", 3)
    rng = np.random.default_rng(3)
    terms = [([(int(q), "XYZ"[int(o)])], complex(c) / 1e5) for q, o, c in
             zip(rng.integers(0, 4, 120000), rng.integers(0, 3, 120000), rng.normal(size=120000))]
    for sim in sims:
        sim.apply_qubit_operator(terms, [0, 1, 2, 3])
    assert np.max(np.abs(sims[0].cheat_numpy()[1] - sims[1].cheat_numpy()[1])) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,count,one_x", [(1, 1, False), (7, 64, False), (7, 65, False), (18, 20, False), (18, 65, False),
                                           (19, 3, False), (20, 2, False), (21, 1, False), (21, 2, True), (21, 2, False)])
def test_gpu_operator_routes(precision, n, count, one_x):
    """With and without tiles, at the edges of both: strings 64 and 65, qubits 18 to 21, one x and two.  The
    coefficients add up to 1, so amplitudes stay below 1 and a string rounds each a few times."""
    sims = simulators(n, precision, n + count)
    rng = np.random.default_rng(n * count)
    terms = []
    for t in range(count):
        ops = [(int(q), "XYZ"[int(o)]) for q, o in zip(range(n), rng.integers(0, 3, size=n))]
        if one_x:
            ops = [(q, "X") for q in range(0, n, 2)] + [(q, "Z") for q in range(1, n, 2) if t or q % 4 == 1]
        terms.append((ops, complex(np.exp(1j * t)) / count))
    for sim in sims:
        sim.apply_qubit_operator(terms, list(range(n)))
    eps = 2.0 ** -53 if precision == "c128" else 2.0 ** -24
    assert np.max(np.abs(sims[0].cheat_numpy()[1] - sims[1].cheat_numpy()[1])) <= 8 * (count * 2.0 ** -53 + eps)
