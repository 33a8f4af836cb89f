"""Expectation values from LDS tiles (projectq_amd/csrc/energy_plan.hpp, energy.hip): the plan against
brute force on the CPU, and the kernels against the oracle at the edges of the tile shapes."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")
CSRC = os.path.join(ROOT, "projectq_amd", "csrc")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("energy") / "libenergy_emu.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, os.path.join(NATIVE, "energy_emu.cpp"),
                    os.path.join(CSRC, "energy_plan.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib).energy_emu


def random_terms(n, count, rng, kind):
    """[(x, z, omega, c)]: Hermitian strings, now and then several with one x, an identity and a
    string that is not Hermitian (it contributes nothing)."""
    out = []
    for _ in range(count):
        x, z = int(rng.integers(0, 1 << n)), int(rng.integers(0, 1 << n))
        if kind == "local":
            x, z = x & (1 << int(rng.integers(0, n))), z & (3 << int(rng.integers(0, n))) & ((1 << n) - 1)
        if out and rng.random() < 0.3:
            x = out[-1][0]
        sign = complex(rng.choice([-1, 1]))
        out.append((x, z, sign * (1j if bin(x & z).count("1") & 1 else 1), float(rng.normal())))
    out[0] = (0, 0, 1 + 0j, 0.7)
    if count > 2:
        out[1] = (1, 1, 1 + 0j, 5.0)  # X Z on one qubit with a real phase
    return out


def expectation(psi, terms):
    i = np.arange(psi.size)
    total = 0.0
    for x, z, omega, c in terms:
        if (bin(x & z).count("1") & 1) != (omega.real == 0):
            continue
        j = i ^ x
        sign = 1 - 2 * np.array([bin(v).count("1") & 1 for v in (j & z)])
        total += c * np.sum(psi.conj() * omega * sign * psi[j]).real
    return total


@pytest.mark.parametrize("c64", [False, True])
@pytest.mark.parametrize("kind", ["random", "local"])
@pytest.mark.parametrize("n,count", [(1, 3), (3, 9), (7, 40), (8, 12), (9, 5), (11, 128), (12, 30), (13, 60), (14, 90)])
def test_plan_equals_brute_force(emu, c64, kind, n, count):
    rng = np.random.default_rng(n * 1000 + count)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi /= np.linalg.norm(psi)
    terms = random_terms(n, count, rng, kind)
    u64 = ctypes.c_ulonglong * count
    dbl = ctypes.c_double
    omega = (dbl * (2 * count))(*[v for t in terms for v in (t[2].real, t[2].imag)])
    out = dbl()
    passes = emu(psi.ctypes.data_as(ctypes.POINTER(dbl)), n, int(c64), u64(*[t[0] for t in terms]), u64(*[t[1] for t in terms]),
                 omega, (dbl * count)(*[t[3] for t in terms]), count, ctypes.byref(out))
    assert passes > 0
    # |<P>| <= 1 for each string; sums of 2^n terms in FP64
    assert abs(out.value - expectation(psi, terms)) <= 1e-14 * sum(abs(t[3]) for t in terms) * n


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,count", [(1, 3), (5, 20), (8, 10), (9, 140), (11, 30), (12, 9), (13, 300), (16, 64)])
def test_gpu_energy_against_oracle(precision, n, count):
    from oracle.cpu_sim import OracleSimulator
    from projectq_amd import Simulator, circuits

    rng = np.random.default_rng(n + count)
    psi = (rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)).astype(np.complex64 if precision == "c64" else np.complex128)
    psi = (psi / np.linalg.norm(psi)).astype(psi.dtype).astype(np.complex128)
    terms = circuits.random_pauli_operator(n, count, 7) + [([], 0.25), ([(0, "Y"), (0, "X")], 0.5), ([(n - 1, "Z")], -1.0)]
    ids = [int(q) for q in rng.permutation(n)]
    values = []
    for sim in (OracleSimulator(1), Simulator(1, precision=precision, capacity_qubits=n)):
        for q in range(n):
            sim.allocate_qubit(q)
        sim.set_wavefunction(psi, list(range(n)))
        values.append(sim.get_expectation_value(terms, ids))
    # the same FP64 products of the same amplitudes, summed in another order
    assert abs(values[0] - values[1]) <= 1e-13 * sum(abs(c) for _, c in terms)
