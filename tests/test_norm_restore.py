"""The complex64 norm guard behind windows that moved qubits: scaling and layout restore in one pass."""

import numpy as np
import pytest

from oracle.cpu_sim import OracleSimulator
from projectq_amd import circuits, commands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12, 15, 17])
def test_scaled_restore(n):
    """Three windows with a read between them: the first read makes the second buffer, the next windows go
    the way under test.  8 roundings of 2^-24 per gate; the norm stays within the guard's budget."""
    from projectq_amd import Simulator

    sim = Simulator(4, precision="c64", fusion="window", planner="tile", capacity_qubits=n)
    sim.set_tile_params(10, 4, 4)
    sim.set_relabel("on")
    ref = OracleSimulator(4)
    gates = 0
    for turn in range(3):
        cmds = circuits.random_layers(n, 8, n // 2, 7 * n + turn, measure=False)
        cmds = [c for c in cmds if turn == 0 or c[0] == "gate"]
        gates += sum(1 for c in cmds if c[0] == "gate")
        for s in (sim, ref):
            commands.execute(s, cmds, gate_fusion=True)
            s.run()
        assert sim.last_plan()["relabels"] > 0
        got, want = np.array(sim.cheat_numpy()[1]), np.array(ref.cheat_numpy()[1])
        assert np.max(np.abs(got - want)) <= 8 * gates * 2.0 ** -24
        # budget 2.5e-7 on the norm, and one rounding per amplitude in the scaling
        assert abs(np.linalg.norm(got) - 1.0) <= 2.5e-7 + 2.0 ** -24
        assert sim.cheat_numpy()[0] == ref.cheat_numpy()[0]
