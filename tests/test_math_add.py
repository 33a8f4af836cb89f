"""Additions of a constant: the source of every destination on the CPU, and every route of the dispatch on the GPU,
against x -> x + a on each register modulo 2^width."""

import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "projectq_amd", "csrc")


def destinations(n, a, regs, ctrl):
    i = np.arange(1 << n, dtype=np.int64)
    on = np.ones(1 << n, dtype=bool)
    for c in ctrl:
        on &= ((i >> c) & 1) == 1
    j = i.copy()
    for reg in regs:
        x = sum((((i >> q) & 1) << b) for b, q in enumerate(reg))
        x = (x + a) & ((1 << len(reg)) - 1)
        for b, q in enumerate(reg):
            j = (j & ~(1 << q)) | (((x >> b) & 1) << q)
    return np.where(on, j, i)


def layouts(n, rng):
    """[(registers, controls)]: neighbours, gaps, descending, mixed, shuffled, with controls."""
    ids = list(range(n))
    out = [([ids], []), ([ids[::-1]], []), ([ids[::2]], [ids[1]]), ([ids[1::2][::-1]], [ids[0]]),
           ([ids[: n // 2], ids[n // 2 :][::-1]], []), ([ids[:1]], ids[1:])]
    if n > 2:
        out.append(([ids[-2:]], [0]))
    for _ in range(4):
        p = rng.sample(ids, n)
        out.append(([sorted(p[: n // 3]), p[n // 3 : 2 * (n // 3)]], p[-1:]))
    return [([r for r in regs if r], ctrl) for regs, ctrl in out if any(regs)]


def test_sources(tmp_path):
    lib = str(tmp_path / "libmath_add_emu.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, os.path.join(ROOT, "tests", "native", "math_add_emu.cpp"),
                    os.path.join(CSRC, "math_map.cpp"), "-o", lib], check=True)
    emu = ctypes.CDLL(lib).math_add_emu
    rng = random.Random(1)
    for n in (2, 3, 7, 10):
        for a in (0, 1, 3, -1, -6, 2**30, 1 << (n - 1)):
            for regs, ctrl in layouts(n, rng):
                in_order = all(r in (sorted(r), sorted(r, reverse=True)) for r in regs)
                flat = [q for r in regs for q in r]
                got = (ctypes.c_uint * (1 << n))()
                ok = emu(ctypes.c_longlong(a), (ctypes.c_uint * len(flat))(*flat), (ctypes.c_uint * len(regs))(*map(len, regs)),
                         len(regs), ctypes.c_ulonglong(sum(1 << c for c in ctrl)), n, got)
                assert bool(ok) == in_order
                if ok:
                    to = destinations(n, a, regs, ctrl)
                    assert np.array_equal(to[np.array(got)], np.arange(1 << n))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c64", "c128"])
@pytest.mark.parametrize("n", [3, 10, 11, 14, 21, 22])
def test_routes(n, precision):
    """From memory order, in tiles (22 qubits: 32 MiB and more), by gather and on the general path; amplitudes
    move, so they stay equal."""
    from projectq_amd import Simulator

    rng = random.Random(n)
    sim = Simulator(1, precision=precision, capacity_qubits=n)
    for q in range(n):
        sim.allocate_qubit(q)
    g = np.random.default_rng(n)
    real = np.float32 if precision == "c64" else np.float64
    psi = g.normal(size=(1 << n, 2)).astype(real).astype(np.float64).view(np.complex128).reshape(-1)
    sim.set_wavefunction(psi, list(range(n)))
    for regs, ctrl in layouts(n, rng):
        a = rng.randint(-50, 50)
        sim._math_op(0, [a], regs, ctrl)
        want = np.empty_like(psi)
        want[destinations(n, a, regs, ctrl)] = psi
        psi = want
        assert np.array_equal(sim.cheat_numpy()[1], psi)
