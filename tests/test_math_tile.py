"""emulate_math in place through LDS tiles: the tile plan against the gather plan on the CPU (register
orders, widths, controls inside and outside the tile), the kernel against the general path's result on the GPU."""

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

CALLS = [
    (F.ADD_CONSTANT, [5], [3]), (F.ADD_CONSTANT, [-3], [2, 3]), (F.ADD_QUANTUM, [], [3, 3]), (F.ADD_QUANTUM, [], [3, 3, 1]),
    (F.ADD_QUANTUM, [], [8, 7]), (F.SUBTRACT_QUANTUM, [], [2, 4]), (F.INVERSE_ADD_QUANTUM, [], [3, 3, 2]),
    (F.COMPARATOR, [], [3, 2, 1]), (F.MULTIPLY_QUANTUM, [], [2, 3, 3]), (F.INVERSE_MULTIPLY_QUANTUM, [], [3, 2, 4]),
    (F.ADD_CONSTANT_MOD_N, [3, 7], [3]), (F.ADD_CONSTANT_MOD_N, [100, 141], [8]),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [7, 15], [4]), (F.MULTIPLY_BY_CONSTANT_MOD_N, [23, 187], [8]),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [5, 4091], [12]),
]


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("math") / "libmath_tile_emu.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, os.path.join(NATIVE, "math_tile_emu.cpp"),
                    os.path.join(CSRC, "math_map.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib).math_tile_emu


def _registers(widths, n, rng, in_order):
    picks = rng.sample(range(n), n)
    regs, at = [], 0
    for w in widths:
        regs.append(sorted(picks[at : at + w]) if in_order else picks[at : at + w])
        at += w
    return regs, picks[at:]


@pytest.mark.parametrize("opcode,params,widths", CALLS)
def test_tile_sources_equal_the_gather(emu, opcode, params, widths):
    rng = random.Random(opcode * 100 + sum(widths))
    seen = set()
    for trial in range(12):
        c64, n_ctrl = trial % 2, (trial // 2) % 4
        n = sum(widths) + n_ctrl + rng.randint(0, 4)
        regs, rest = _registers(widths, n, rng, in_order=trial % 3 != 0)
        a, N = (list(params) + [0, 1])[:2] if params else (0, 1)
        flat = [q for r in regs for q in r]
        got = emu(opcode, ctypes.c_longlong(a), ctypes.c_longlong(N), (ctypes.c_uint * len(flat))(*flat),
                  (ctypes.c_uint * len(regs))(*map(len, regs)), len(regs),
                  ctypes.c_ulonglong(sum(1 << q for q in rest[:n_ctrl])), n, c64)
        assert got != 3, (regs, rest[:n_ctrl], n, c64)
        seen.add(got)
    assert 2 in seen or widths == [12]


@pytest.mark.gpu
@pytest.mark.parametrize("n_ctrl", [0, 1, 3])
@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("opcode,params,widths,n", [
    (F.ADD_CONSTANT, [5], [3], 7),
    (F.ADD_QUANTUM, [], [4, 4], 11),            # exactly a complex128 tile
    (F.ADD_QUANTUM, [], [5, 4, 1], 13),
    (F.MULTIPLY_QUANTUM, [], [3, 4, 6], 16),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [23, 187], [8], 14),
    (F.MULTIPLY_BY_CONSTANT_MOD_N, [5, 4091], [12], 15),  # beyond a complex128 tile
    (F.ADD_CONSTANT_MOD_N, [100, 37], [8], 15),           # up to seven sources
])
def test_gpu_moves_amplitudes_exactly(precision, opcode, params, widths, n, n_ctrl):
    from projectq_amd import Simulator

    rng = random.Random(n * 10 + n_ctrl)
    n = max(n, sum(widths) + n_ctrl)
    regs, rest = _registers(widths, n, rng, in_order=True)
    ctrl = rest[:n_ctrl]
    g = np.random.default_rng(n)
    real = np.float32 if precision == "c64" else np.float64
    psi = g.normal(size=(1 << n, 2)).astype(real).astype(np.float64).view(np.complex128).reshape(-1)
    sim = Simulator(1, precision=precision, capacity_qubits=n)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction(psi, list(range(n)))
    sim._math_op(opcode, params, regs, ctrl)
    index = np.arange(1 << n)
    on = np.all([(index >> c) & 1 for c in ctrl], axis=0) if ctrl else np.ones(1 << n, dtype=bool)
    to = index.copy()
    for i in index[on]:
        values = [sum(((int(i) >> q) & 1) << b for b, q in enumerate(r)) for r in regs]
        j = int(i)
        for r, v in zip(regs, F.apply_op(opcode, params, [len(r) for r in regs], values)):
            for b, q in enumerate(r):
                j = (j & ~(1 << q)) | (((v >> b) & 1) << q)
        to[i] = j
    want = np.zeros_like(psi)
    np.add.at(want, to, psi)  # in index order, as the reference adds
    want = want.view(np.float64).astype(real).astype(np.float64).view(np.complex128)
    assert np.array_equal(sim.cheat_numpy()[1], want)
