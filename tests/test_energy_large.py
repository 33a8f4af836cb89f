"""Energies of states beyond the caches, where the tiles have shorter segments: against numpy in 64 bits.

The products and sums are FP64 on the stored amplitudes: 2^24 terms of a normalised state, each string within
2^24 * 2^-53 of exact in the worst case, far less pairwise."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,terms", [(24, "c64", 7), (24, "c64", 8), (23, "c128", 9)])
def test_energy_against_numpy(n, precision, terms):
    from projectq_amd import Simulator

    rng = np.random.default_rng(n + terms)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi /= np.linalg.norm(psi)
    if precision == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    ham = []
    for _ in range(terms):
        ops = rng.integers(0, 4, size=n)
        ham.append(([(q, "IXYZ"[o]) for q, o in enumerate(ops) if o], float(rng.normal())))
    sim = Simulator(1, precision=precision, capacity_qubits=n)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction(psi, list(range(n)))
    got = sim.get_expectation_value(ham, list(range(n)))
    index, want = np.arange(1 << n, dtype=np.uint32), 0.0
    for ops, c in ham:
        x = np.uint32(sum(1 << q for q, p in ops if p in "XY"))
        z = np.uint32(sum(1 << q for q, p in ops if p in "YZ"))
        source = index ^ x
        odd = source & z
        for shift in (16, 8, 4, 2, 1):
            odd ^= odd >> np.uint32(shift)
        image = psi[source]
        image[(odd & 1) == 1] *= -1.0
        want += c * (np.vdot(psi, image) * 1j ** sum(p == "Y" for _, p in ops)).real
    assert abs(got - want) <= 2.0 ** 24 * 2.0 ** -53 * sum(abs(c) for _, c in ham)
