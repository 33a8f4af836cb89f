"""The gather form of emulate_math (projectq_amd/csrc/math_map.hpp) against the forward map of every
function it covers: register orders, widths, controls and constants, every basis state."""

import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

from projectq_amd import _mathfuncs as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")
CSRC = os.path.join(ROOT, "projectq_amd", "csrc")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("math") / "libmath_emu.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, os.path.join(NATIVE, "math_emu.cpp"),
                    os.path.join(CSRC, "math_map.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib).math_emu


def plan(emu, opcode, params, regs, ctrl, n, c64=False):
    """{destination: [sources]} of the plan, or None where it does not cover the call."""
    a, N = (list(params) + [0, 1])[:2] if params else (0, 1)
    flat = [q for r in regs for q in r]
    first, visited = (ctypes.c_uint * ((1 << n) + 1))(), (ctypes.c_uint * (1 << n))()
    sources = (ctypes.c_uint * (4 << n))()
    got = emu(opcode, ctypes.c_longlong(a), ctypes.c_longlong(N), (ctypes.c_uint * len(flat))(*flat),
              (ctypes.c_uint * len(regs))(*map(len, regs)), len(regs),
              ctypes.c_ulonglong(sum(1 << q for q in ctrl)), n, int(c64), first, sources, visited)
    if got == 0:
        return None
    assert got == 1
    assert sorted(visited) == list(range(1 << n))  # every destination once
    return {i: list(sources[first[i] : first[i + 1]]) for i in range(1 << n)}


def forward(opcode, params, regs, ctrl, n):
    """{destination: [sources in index order]} of the reference's loop (simulator.hpp:246-265)."""
    out = {i: [] for i in range(1 << n)}
    for i in range(1 << n):
        j = i
        if all((i >> c) & 1 for c in ctrl):
            vals = [sum(((i >> q) & 1) << b for b, q in enumerate(r)) for r in regs]
            new = F.apply_op(opcode, params, [len(r) for r in regs], vals)
            for r, v in zip(regs, new):
                for b, q in enumerate(r):
                    j = (j & ~(1 << q)) | (((v >> b) & 1) << q)
        out[j].append(i)
    return out


ONE_TO_ONE = [
    (F.ADD_CONSTANT, [5], [3]), (F.ADD_CONSTANT, [-3], [2, 3]), (F.ADD_CONSTANT, [7], [1, 2, 3]),
    (F.ADD_QUANTUM, [], [3, 3]), (F.ADD_QUANTUM, [], [4, 2]), (F.ADD_QUANTUM, [], [1, 1]),
    (F.ADD_QUANTUM, [], [3, 3, 1]), (F.ADD_QUANTUM, [], [3, 2, 2]),
    (F.SUBTRACT_QUANTUM, [], [3, 3]), (F.SUBTRACT_QUANTUM, [], [2, 4]),
    (F.INVERSE_ADD_QUANTUM, [], [3, 3]), (F.INVERSE_ADD_QUANTUM, [], [3, 3, 2]),
    (F.COMPARATOR, [], [3, 2, 1]), (F.COMPARATOR, [], [1, 4, 1]),
    (F.MULTIPLY_QUANTUM, [], [2, 3, 3]), (F.INVERSE_MULTIPLY_QUANTUM, [], [3, 2, 4]),
]
RESIDUES = [
    (F.ADD_CONSTANT_MOD_N, [3, 7], [3]), (F.ADD_CONSTANT_MOD_N, [9, 5], [5]), (F.ADD_CONSTANT_MOD_N, [0, 3], [2]),
    (F.ADD_CONSTANT_MOD_N, [6, 16], [4]), (F.MULTIPLY_BY_CONSTANT_MOD_N, [3, 7], [3]),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [7, 15], [4]), (F.MULTIPLY_BY_CONSTANT_MOD_N, [22, 15], [5]),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [2, 5], [5]), (F.MULTIPLY_BY_CONSTANT_MOD_N, [1, 2], [1]),
]


@pytest.mark.parametrize("opcode,params,widths", ONE_TO_ONE + RESIDUES)
def test_sources_equal_the_forward_map(emu, opcode, params, widths):
    rng = random.Random(opcode * 100 + sum(widths))
    for trial in range(6):
        n_ctrl = trial % 3
        n = sum(widths) + n_ctrl + rng.randint(0, 2)
        picks = list(range(n)) if trial == 0 else rng.sample(range(n), n)
        regs, at = [], 0
        for w in widths:
            regs.append(picks[at : at + w])
            at += w
        ctrl = picks[at : at + n_ctrl]
        got = plan(emu, opcode, params, regs, ctrl, n, c64=trial % 2 == 1)
        want = forward(opcode, params, regs, ctrl, n)
        if got is None:
            # only residues on a register out of significance order, three sources or more
            assert opcode in (F.ADD_CONSTANT_MOD_N, F.MULTIPLY_BY_CONSTANT_MOD_N) and regs[0] != sorted(regs[0])
            assert max(map(len, want.values())) > 2
            continue
        for i in range(1 << n):
            assert got[i] == want[i] or (len(want[i]) == 2 and sorted(got[i]) == want[i])


@pytest.mark.parametrize("opcode,params,regs,ctrl", [
    (F.ADD_QUANTUM, [], [[0, 1], [2, 3, 4]], []),          # wider second register: sums collide
    (F.ADD_QUANTUM, [], [[0, 1], [1, 2]], []),             # a shared qubit
    (F.ADD_QUANTUM, [], [[0, 1], [2, 3]], [1]),            # a control inside a register
    (F.COMPARATOR, [], [[0], [1], [2, 3]], []),            # the result bit is a wider register
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [3, 6], [[0, 1, 2]], []),       # not a unit
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [-1, 7], [[0, 1, 2]], []),      # negative residues in C++
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [2**30, 7], [[0, 1, 2]], []),   # the product wraps
    (F.ADD_CONSTANT_MOD_N, [1, 9], [[0, 1, 2]], []),               # N beyond the register
    (F.ADD_CONSTANT_MOD_N, [1, -7], [[0, 1, 2]], []),
    (F.ADD_CONSTANT_MOD_N, [1, 3], [[0, 1], [2, 3]], []),
    (F.DIVIDE_QUANTUM, [], [[0, 1], [2, 3], [4, 5]], []),
])
def test_other_calls_keep_the_general_path(emu, opcode, params, regs, ctrl):
    assert plan(emu, opcode, params, regs, ctrl, 6) is None


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("opcode,params,widths,n", [
    (F.ADD_QUANTUM, [], [3, 3], 6),            # fewer amplitudes than a workgroup
    (F.ADD_QUANTUM, [], [6, 6, 1], 13),        # two workgroups
    (F.ADD_QUANTUM, [], [7, 7], 16),
    (F.INVERSE_ADD_QUANTUM, [], [4, 4, 1], 12),
    (F.MULTIPLY_QUANTUM, [], [3, 4, 6], 14),
    (F.COMPARATOR, [], [5, 6, 1], 12),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [23, 187], [8], 13),
    (F.ADD_CONSTANT_MOD_N, [100, 37], [8], 15),  # up to seven sources
])
def test_gpu_gather_moves_amplitudes_exactly(precision, opcode, params, widths, n):
    from projectq_amd import Simulator

    rng = random.Random(n)
    picks = rng.sample(range(n), n)
    regs, at = [], 0
    for w in widths:
        regs.append(sorted(picks[at : at + w]))
        at += w
    ctrl = picks[at : at + 1] if at < n else []
    g = np.random.default_rng(n)
    real = np.float32 if precision == "c64" else np.float64
    psi = g.normal(size=(1 << n, 2)).astype(real).astype(np.float64).view(np.complex128).reshape(-1)
    sim = Simulator(1, precision=precision, capacity_qubits=n)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction(psi, list(range(n)))
    sim._math_op(opcode, params, regs, ctrl)
    want = np.zeros_like(psi)
    for j, sources in forward(opcode, params, regs, ctrl, n).items():
        for i in sources:
            want[j] += psi[i]
    want = want.view(np.float64).astype(real).astype(np.float64).view(np.complex128)
    assert np.array_equal(sim.cheat_numpy()[1], want)
