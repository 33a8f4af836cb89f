"""Energies of states beyond the caches, where the tiles have shorter segments: against torch in 64 bits.

The products and sums are FP64 on the stored amplitudes: 2^24 terms of a normalised state, each string within
2^24 * 2^-53 of exact in the worst case, far less pairwise."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,terms", [(23, "c64", 12), (24, "c64", 7), (24, "c64", 8), (24, "c64", 30), (23, "c128", 20)])
def test_energy_against_torch(n, precision, terms):
    import numpy as np
    import torch

    from projectq_amd import Simulator

    gen = torch.Generator(device="cuda").manual_seed(n + terms)
    real = torch.float32 if precision == "c64" else torch.float64
    psi = torch.randn(1 << n, 2, generator=gen, device="cuda", dtype=real)
    psi = torch.view_as_complex(psi.div_(float(psi.double().square().sum()) ** 0.5))
    rng = np.random.default_rng(n)
    ham = []
    for _ in range(terms):
        ops = rng.integers(0, 4, size=n)
        ham.append(([(q, "IXYZ"[o]) for q, o in enumerate(ops) if o], float(rng.normal())))
    sim = Simulator(1, precision=precision, capacity_qubits=n)
    for q in range(n):
        sim.allocate_qubit(q)
    sim.set_wavefunction_device(psi, list(range(n)))
    got = sim.get_expectation_value(ham, list(range(n)))
    wide, index, want = psi.to(torch.complex128), torch.arange(1 << n, device="cuda"), 0.0
    for ops, c in ham:
        x = sum(1 << q for q, p in ops if p in "XY")
        z = sum(1 << q for q, p in ops if p in "YZ")
        source = index ^ x
        sign = source & z
        for shift in (32, 16, 8, 4, 2, 1):
            sign = sign ^ (sign >> shift)
        image = wide[source] * (1.0 - 2.0 * (sign & 1).double()) * (1j ** sum(p == "Y" for _, p in ops))
        want += c * float((wide.conj() * image).real.sum())
    assert abs(got - want) <= 2.0 ** 24 * 2.0 ** -53 * sum(abs(c) for _, c in ham)
