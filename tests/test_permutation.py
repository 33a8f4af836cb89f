"""Qubit layout permutations through LDS tiles: plan and index rules on the CPU, the kernel on the GPU."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle.cpu_sim import OracleSimulator
from projectq_amd import circuits, commands

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "native", "_build", "libperm_emu.so")


@pytest.fixture(scope="module")
def emu():
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    csrc = os.path.join(ROOT, "projectq_amd", "csrc")
    srcs = [os.path.join(ROOT, "tests", "native", "perm_emu.cpp"), os.path.join(csrc, "planner.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", csrc, *srcs, "-o", LIB], check=True)
    return ctypes.CDLL(LIB)


@pytest.mark.parametrize("c64", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 8, 9, 11, 12, 13, 15, 17])
def test_planned_permutation(emu, n, c64):
    rng = np.random.default_rng(n)
    orders = [np.arange(n), np.arange(n)[::-1], np.roll(np.arange(n), 1), *(rng.permutation(n) for _ in range(4))]
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    for to in orders:
        to = np.ascontiguousarray(to, dtype=np.uint32)
        src = np.arange(1 << n, dtype=np.uint32)
        dst, conflicts = np.zeros_like(src), np.zeros(2, dtype=np.uint32)
        assert emu.perm_run(n, ptr(to), c64, ptr(src), ptr(dst), ptr(conflicts)) == 0
        want = np.zeros_like(src)
        image = np.zeros_like(src)
        for p in range(n):
            image |= ((src >> p) & 1) << to[p]
        want[image] = src
        assert np.array_equal(dst, want)
        if n >= 11:  # free of bank conflicts on both sides
            assert conflicts.max() == 1, (list(to), list(conflicts))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c64", "c128"])
@pytest.mark.parametrize("n", [11, 12, 13, 16, 19])
def test_layout_restored(n, precision):
    """Windows with relabelling leave another layout; reading the state restores it.  Rounding: 8 per gate
    (2^-24 or 2^-53) on amplitudes of at most 1."""
    from projectq_amd import Simulator

    cmds = circuits.random_layers(n, 6, n // 2, n, measure=False)
    sim = Simulator(4, precision=precision, fusion="window", planner="tile", capacity_qubits=n)
    sim.set_tile_params(10, 4, 4)
    sim.set_relabel("on")
    ref = OracleSimulator(4)
    for s in (sim, ref):
        commands.execute(s, cmds, gate_fusion=True)
        s.run()
    assert sim.last_plan()["relabels"] > 0
    gates = sum(1 for c in cmds if c[0] == "gate")
    eps = 2.0 ** -24 if precision == "c64" else 2.0 ** -53
    assert np.max(np.abs(np.array(sim.cheat_numpy()[1]) - np.array(ref.cheat_numpy()[1]))) <= 8 * gates * eps
