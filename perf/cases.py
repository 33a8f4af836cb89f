"""What a program does with this simulator, as timed cases.

`listed()` names the cases, `draw(rng)` gives one more of the same ranges, `prepare(case, seed)` builds
what the program holds before the call, `run(state)` is one pass through the public entry points
and returns its outputs, `work(case)` is what one pass cannot do without, and `exact(case, seed)`
is the result in 64 bits from plain torch.

Kinds:

* gates    -- a circuit on a resident state.  Its mode is the reference's default (`default`: run()
              after every gate), its gate fusion (`fusion`: blocks of up to 5 qubits) or the
              window queue under the learned planner (`window`).  Circuits: random layers (H, a
              rotation per qubit, CNOTs on random pairs), QFT followed by rotations and controlled
              rotations, and mixed 1/2/3-qubit gates.
* vqe      -- one evaluation of a variational energy as a ProjectQ program does it: allocate, ansatz,
              flush, expectation value, measure, deallocate.
* energy   -- expectation value of a Hamiltonian on a resident state.
* evolve   -- time evolution under a Hamiltonian.
* add      -- AddQuantum on two registers through emulate_math.
* modexp   -- the controlled multiplications modulo N of order finding.
* readout  -- probabilities of a few bit patterns, then every qubit measured one by one.
* batch    -- the energies of many small ansatze in one graph launch.
"""

import math

import numpy as np
import torch

DEVICE = "cuda"


# ---------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest calls: one step of a variational loop on a few qubits, latency and launches
        dict(name="vqe_10q", kind="vqe", n=10, layers=4, terms=30, precision="c128"),
        # the reference's gate_fusion=True on a medium register
        dict(name="gates_fusion_21q", kind="gates", circuit="layers", mode="fusion", n=21, depth=5, precision="c128"),
        # a general circuit in single precision: 1-, 2- and 3-qubit gates through the planner
        dict(name="gates_mixed_23q", kind="gates", circuit="mixed", mode="window", n=23, depth=20, precision="c64"),
        # the reference's precision through the planner: QFT and controlled rotations
        dict(name="gates_qft_27q", kind="gates", circuit="qft", mode="window", n=27, depth=5, precision="c128"),
        # five layers of the random-layer circuit on a large single-precision state
        dict(name="gates_layers_30q", kind="gates", circuit="layers", mode="window", n=30, depth=5, precision="c64"),
        # a Hamiltonian of 100 random strings on a state that fits the caches
        dict(name="energy_20q", kind="energy", n=20, terms=100, hamiltonian="random", precision="c128"),
        # the same on a state far beyond the caches
        dict(name="energy_28q", kind="energy", n=28, terms=40, hamiltonian="random", precision="c64"),
        # a quench of a transverse-field Ising chain
        dict(name="evolve_21q", kind="evolve", n=21, hamiltonian="ising", time=0.1, controls=0, precision="c128"),
        # b <- a + b on two 14-bit registers in superposition
        dict(name="add_28q", kind="add", n=28, precision="c64"),
        # order finding modulo an 8-bit number: 14 controlled multiplications
        dict(name="modexp_22q", kind="modexp", n=22, bits=8, precision="c128"),
        # the end of a program: 8 probabilities, then All(Measure)
        dict(name="readout_27q", kind="readout", n=27, queries=8, precision="c64"),
        # variational batch: one graph launch for 160 circuits of 10 to 18 qubits, 100 strings each
        dict(name="batch_160", kind="batch", circuits=160, lo=10, hi=18, layers=6, terms=100, precision="c64"),
    ]


def draw(rng):
    precision = rng.choice(["c64", "c128"])
    less = 1 if precision == "c128" else 0  # twice the bytes: one qubit fewer
    kind = rng.choice(["gates", "gates", "gates", "gates", "vqe", "energy", "energy", "evolve", "add", "modexp",
                       "readout", "batch"])
    if kind == "gates":
        mode = rng.choice(["default", "fusion", "window", "window"])
        circuit = rng.choice(["layers", "mixed", "qft"])
        n = rng.randint(6, {"default": 25, "fusion": 27, "window": 29}[mode] - less)
        depth = {"layers": rng.randint(1, 5), "mixed": rng.randint(4, 20), "qft": rng.randint(1, 5)}[circuit]
        return dict(kind=kind, circuit=circuit, mode=mode, n=n, depth=depth, precision=precision)
    if kind == "vqe":
        return dict(kind=kind, n=rng.randint(4, 14), layers=rng.randint(1, 6), terms=rng.randint(5, 60),
                    precision="c128")
    if kind == "energy":
        ham = rng.choice(["random", "ising", "heisenberg"])
        return dict(kind=kind, n=rng.randint(10, 28 - less), terms=rng.randint(5, 100), hamiltonian=ham,
                    precision=precision)
    if kind == "evolve":
        return dict(kind=kind, n=rng.randint(8, 22 - less), hamiltonian=rng.choice(["ising", "heisenberg", "random"]),
                    time=round(rng.uniform(0.02, 0.12), 3), controls=rng.randint(0, 1), precision="c128")
    if kind == "add":
        return dict(kind=kind, n=rng.randint(12, 28 - less), precision=precision)
    if kind == "modexp":
        bits = rng.randint(4, 10)
        return dict(kind=kind, n=rng.randint(bits + 3, 22), bits=bits, precision=precision)
    if kind == "readout":
        return dict(kind=kind, n=rng.randint(10, 28 - less), queries=rng.randint(1, 12), precision=precision)
    lo = rng.randint(6, 11)
    return dict(kind=kind, circuits=int(2 ** rng.uniform(3, 7)), lo=lo, hi=rng.randint(lo, 16), layers=rng.randint(2, 6),
                terms=rng.randint(10, 100), precision=precision)


# ---------------------------------------------------------------------------- circuits and Hamiltonians
H = np.array([[1, 1], [1, -1]], dtype=np.complex128) / math.sqrt(2.0)
X = np.array([[0, 1], [1, 0]], dtype=np.complex128)
SWAP = np.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], dtype=np.complex128)


def _rotation(axis, a):
    c, s = math.cos(a / 2), math.sin(a / 2)
    if axis == 0:
        return np.array([[c, -1j * s], [-1j * s, c]], dtype=np.complex128)
    if axis == 1:
        return np.array([[c, -s], [s, c]], dtype=np.complex128)
    return np.array([[c - 1j * s, 0], [0, c + 1j * s]], dtype=np.complex128)


def _phase(a):
    return np.array([[1, 0], [0, complex(math.cos(a), math.sin(a))]], dtype=np.complex128)


def _rzz(a):
    m, p = complex(math.cos(a / 2), -math.sin(a / 2)), complex(math.cos(a / 2), math.sin(a / 2))
    return np.diag([m, p, p, m]).astype(np.complex128)


def _circuit(case, seed):
    """Commands of projectq_amd.commands: ("gate", matrix, targets, controls)."""
    rng = np.random.default_rng(seed)
    n, depth, out = case["n"], case["depth"], []

    def add(m, targets, controls=()):
        out.append(("gate", m, tuple(int(t) for t in targets), tuple(sorted(int(c) for c in controls))))

    def rotations():
        kinds, angles = rng.integers(0, 3, size=n), rng.uniform(0.0, 2.0 * math.pi, size=n)
        for q in range(n):
            add(_rotation(kinds[q], angles[q]), [q])

    if case["circuit"] == "layers":
        for _ in range(depth):
            for q in range(n):
                add(H, [q])
            rotations()
            for _ in range(n // 2):
                c, t = rng.choice(n, size=2, replace=False)
                add(X, [t], [c])
    elif case["circuit"] == "qft":
        for i in range(n):
            add(H, [n - 1 - i])
            for j in range(n - 1 - i):
                add(_phase(math.pi / (1 << (1 + j))), [n - 1 - i], [n - 2 - j - i])
        for _ in range(depth):
            rotations()
            for _ in range(n // 2):
                k = int(rng.integers(1, 4))
                picks = rng.choice(n, size=k + 1, replace=False)
                add(_rotation(2, rng.uniform(0.0, 2.0 * math.pi)), [picks[0]], picks[1:])
    else:
        for _ in range(depth):
            perm, i = rng.permutation(n), 0
            while i < n:
                width = min(int(rng.choice([1, 2, 3], p=[0.5, 0.35, 0.15])), n - i)
                q, a, k = perm[i : i + width], rng.uniform(0.0, 2.0 * math.pi), int(rng.integers(0, 12))
                i += width
                if width == 1:
                    add(_rotation(k % 3, a), q)
                elif width == 2:
                    if k % 4 == 0:
                        add(X, [q[1]], [q[0]])
                    elif k % 4 == 1:
                        add(_phase(a), [q[1]], [q[0]])
                    elif k % 4 == 2:
                        add(_rzz(a), q)
                    else:
                        add(SWAP, q)
                elif k % 2 == 0:
                    add(X, [q[2]], q[:2])
                else:
                    add(SWAP, q[1:], [q[0]])
    return out


def _ansatz(n, layers, rng):
    out = []
    for _ in range(layers):
        th = rng.uniform(0.0, 2.0 * math.pi, size=(n, 2))
        for q in range(n):
            out.append(("gate", _rotation(1, th[q, 0]), (q,), ()))
            out.append(("gate", _rotation(2, th[q, 1]), (q,), ()))
        for q in range(n - 1):
            out.append(("gate", X, (q + 1,), (q,)))
    return out


def _hamiltonian(kind, n, terms, rng):
    """[(list of (qubit, 'X'|'Y'|'Z'), real coefficient)], the backend's term format."""
    out = []
    if kind == "random":  # each qubit I, X, Y or Z
        for _ in range(terms):
            ops = rng.integers(0, 4, size=n)
            out.append(([(q, "IXYZ"[o]) for q, o in enumerate(ops) if o], float(rng.normal())))
    elif kind == "ising":  # transverse field on an open chain
        out += [([(q, "Z"), (q + 1, "Z")], float(rng.normal())) for q in range(n - 1)]
        out += [([(q, "X")], float(rng.normal())) for q in range(n)]
    else:
        for q in range(n - 1):
            out += [([(q, p), (q + 1, p)], float(rng.normal())) for p in "XYZ"]
        out += [([(q, "Z")], float(rng.normal())) for q in range(n)]
    return out


def _state(case, seed):
    """A normalised random state of the case's precision, on the GPU."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    real = torch.float32 if case["precision"] == "c64" else torch.float64
    psi = torch.randn(1 << case["n"], 2, generator=g, device=DEVICE, dtype=real)
    if case["kind"] == "modexp":  # the work register holds residues modulo N only
        value = torch.arange(1 << case["n"], device=DEVICE) & ((1 << case["bits"]) - 1)
        psi[value >= _modulus(case, seed)[0]] = 0
    norm = math.sqrt(float(psi.double().square().sum()))
    return torch.view_as_complex(psi.div_(norm))


def _modulus(case, seed):
    """(odd N of `bits` bits, a coprime to it)."""
    rng = np.random.default_rng(seed)
    bits = case["bits"]
    N = int(rng.integers(1 << (bits - 2), 1 << (bits - 1))) * 2 + 1
    while True:
        a = int(rng.integers(2, N))
        if math.gcd(a, N) == 1:
            return N, a


def _terms_of(case, seed):
    return _hamiltonian(case["hamiltonian"], case["n"] - case.get("controls", 0), case.get("terms", 12),
                        np.random.default_rng(seed + 1))


def _batch_of(case, seed):
    rng = np.random.default_rng(seed)
    sizes = [int(v) for v in rng.integers(case["lo"], case["hi"] + 1, size=case["circuits"])]
    return ([(n, _ansatz(n, case["layers"], rng)) for n in sizes],
            [_hamiltonian("random", n, case["terms"], rng) for n in sizes])


def _queries(case, seed):
    rng = np.random.default_rng(seed + 2)
    n = case["n"]
    out = []
    for _ in range(case["queries"]):
        ids = [int(q) for q in rng.choice(n, size=min(n, 8), replace=False)]
        out.append(([bool(v) for v in rng.integers(0, 2, size=len(ids))], ids))
    return out


# ---------------------------------------------------------------------------- what a program holds
def _simulator(case, seed, load=True):
    from projectq_amd import Simulator

    mode = case.get("mode", "default")
    kw = dict(fusion="window", planner="learned") if mode == "window" else {}
    sim = Simulator(seed & 0xFFFFFFFF, precision=case["precision"], capacity_qubits=case["n"], **kw)
    if load:
        for q in range(case["n"]):
            sim.allocate_qubit(q)
        sim.set_wavefunction_device(_state(case, seed), list(range(case["n"])))
    return sim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        from projectq_amd.batch import BatchExpectation

        circuits, operators = _batch_of(case, seed)
        return dict(case=case, batch=BatchExpectation(circuits, operators, precision=case["precision"]))
    if kind == "vqe":
        rng = np.random.default_rng(seed)
        return dict(case=case, sim=_simulator(case, seed, load=False), gates=_ansatz(case["n"], case["layers"], rng),
                    terms=_hamiltonian("random", case["n"], case["terms"], rng))
    state = dict(case=case, sim=_simulator(case, seed))
    if kind == "gates":
        state["gates"] = _circuit(case, seed)
    elif kind in ("energy", "evolve"):
        state["terms"] = _terms_of(case, seed)
    elif kind == "add":
        from projectq_amd import gates

        n, half = case["n"], case["n"] // 2
        state["add"] = gates.add_quantum(half)
        state["registers"] = [list(range(half)), list(range(n - half, n))]
    elif kind == "modexp":
        N, a = _modulus(case, seed)
        state["N"] = N
        state["factors"] = [pow(a, 1 << k, N) for k in range(case["n"] - case["bits"])]
    elif kind == "readout":
        state["psi"], state["queries"] = _state(case, seed), _queries(case, seed)
    return state


def _amplitudes(sim):
    return torch.as_tensor(sim.device_state()[1], device=DEVICE)


def run(state):
    from projectq_amd import commands

    case = state["case"]
    kind, n = case["kind"], case.get("n")
    if kind == "batch":
        return state["batch"].run()[0]
    sim = state["sim"]
    if kind == "gates":
        commands.execute(sim, state["gates"], gate_fusion=case["mode"] != "default")
        sim.run()
        return _amplitudes(sim)
    if kind == "vqe":
        ids = list(range(n))
        commands.execute(sim, [("allocate", q) for q in ids] + state["gates"] + [("flush",)])
        energy = sim.get_expectation_value(state["terms"], ids)
        bits = commands.execute(sim, [("measure", q) for q in ids] + [("deallocate", q) for q in ids])
        return energy, [bits[q] for q in ids]
    if kind == "energy":
        return sim.get_expectation_value(state["terms"], list(range(n)))
    if kind == "evolve":
        k = case["controls"]
        sim.emulate_time_evolution(state["terms"], case["time"], list(range(n - k)), list(range(n - k, n)))
        return _amplitudes(sim)
    if kind == "add":
        sim.emulate_math(state["add"], state["registers"], [])
        return _amplitudes(sim)
    if kind == "modexp":
        register = list(range(case["bits"]))
        for k, factor in enumerate(state["factors"]):
            sim.emulate_math_multiplyByConstantModN(factor, state["N"], [register], [case["bits"] + k])
        return _amplitudes(sim)
    # readout: the state comes from elsewhere in the program; measuring consumes it
    sim.set_wavefunction_device(state["psi"], list(range(n)))
    chances = [sim.get_probability(bits, ids) for bits, ids in state["queries"]]
    outcomes = [sim.measure_qubits([q])[0] for q in range(n)]
    return chances, outcomes, _amplitudes(sim)


# ---------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    size = 8 if case["precision"] == "c64" else 16
    if kind == "batch":  # states are made and consumed inside the call; the arithmetic is the work
        mid = 0.5 * (case["lo"] + case["hi"])
        amps = case["circuits"] * 2.0 ** mid
        return {"bytes": 2.0 * size * amps, "flops": amps * (case["layers"] * mid * 20 + 8 * case["terms"])}
    amps = 2.0 ** case["n"]
    if kind == "gates":
        # each gate: 2^n amplitudes, halved by each control, a 2^k row each
        flops = sum(amps / 2 ** len(c) * (8 * 2 ** len(t) - 2) for _, _, t, c in _circuit(case, 1))
        return {"bytes": 2 * size * amps, "flops": flops}
    if kind == "vqe":
        return {"bytes": 2 * size * amps, "flops": amps * (case["layers"] * case["n"] * 20 + 8 * case["terms"])}
    if kind == "energy":
        return {"bytes": size * amps, "flops": 8 * amps * len(_terms_of(case, 1))}
    if kind == "evolve":  # one application of the Hamiltonian per Taylor term, at least a dozen
        return {"bytes": 2 * size * amps, "flops": 12 * 8 * amps * len(_terms_of(case, 1))}
    if kind == "readout":  # the state in, read for the first outcome, and out
        return {"bytes": 3 * size * amps, "flops": 8 * amps}
    return {"bytes": 2 * size * amps, "flops": 0.0}


# ---------------------------------------------------------------------------- the result in 64 bits
def _apply(psi, n, m, targets, controls):
    """One gate on a complex128 state vector, in place."""
    view = psi.view([2] * n)
    at = [slice(None)] * n  # axis n - 1 - q is qubit q
    for c in controls:
        at[n - 1 - c] = 1
    parts = []
    for j in range(1 << len(targets)):
        here = list(at)
        for bit, t in enumerate(targets):
            here[n - 1 - t] = (j >> bit) & 1
        parts.append(view[tuple(here)])
    old = [p.clone() for p in parts]
    for r, p in enumerate(parts):
        total = None
        for c, o in enumerate(old):
            if m[r, c] != 0:
                term = o * complex(m[r, c])
                total = term if total is None else total.add_(term)
        p.copy_(total) if total is not None else p.zero_()


def _string(psi, index, ops):
    """A Pauli string applied to a complex128 state vector."""
    x = z = 0
    for q, p in ops:
        x |= (p in "XY") << q
        z |= (p in "YZ") << q
    source = index ^ x
    sign = source & z
    for shift in (32, 16, 8, 4, 2, 1):
        sign = sign ^ (sign >> shift)
    sign = 1.0 - 2.0 * (sign & 1).double()
    return psi[source] * sign * (1j ** sum(p == "Y" for _, p in ops))


def _energy(psi, terms):
    index = torch.arange(psi.numel(), device=psi.device)
    return math.fsum(c * float(torch.sum((psi.conj() * _string(psi, index, ops)).real)) for ops, c in terms)


def exact(case, seed):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "readout" or n > 28:  # measured outcomes are drawn; the largest circuit takes too long
        return None
    if kind == "batch":
        circuits, operators = _batch_of(case, seed)
        out = []
        for (k, gates), terms in zip(circuits, operators):
            psi = torch.zeros(1 << k, dtype=torch.complex128, device=DEVICE)
            psi[0] = 1
            for _, m, t, c in gates:
                _apply(psi, k, m, t, c)
            out.append(_energy(psi, terms))
        return np.array(out)
    if kind == "vqe":
        rng = np.random.default_rng(seed)
        gates, psi = _ansatz(n, case["layers"], rng), torch.zeros(1 << n, dtype=torch.complex128, device=DEVICE)
        psi[0] = 1
        for _, m, t, c in gates:
            _apply(psi, n, m, t, c)
        return _energy(psi, _hamiltonian("random", n, case["terms"], rng)), None
    psi = _state(case, seed).to(torch.complex128)
    if kind == "gates":
        for _, m, t, c in _circuit(case, seed):
            _apply(psi, n, m, t, c)
        return psi
    if kind == "energy":
        return _energy(psi, _terms_of(case, seed))
    index = torch.arange(1 << n, device=DEVICE)
    if kind == "evolve":
        terms, rest = _terms_of(case, seed), psi.clone()
        on = None
        if case["controls"]:
            on = (index >> (n - case["controls"])) == (1 << case["controls"]) - 1
            rest = torch.where(on, psi, torch.zeros_like(psi))
        steps = max(1, math.ceil(case["time"] * sum(abs(c) for _, c in terms)))
        total = rest.clone()
        for _ in range(steps):
            term = total.clone()
            for k in range(1, 40):
                image = torch.zeros_like(term)
                for ops, c in terms:
                    image.add_(_string(term, index, ops), alpha=c)
                term = image * (-1j * case["time"] / steps / k)
                total = total + term
                if float(torch.linalg.vector_norm(term)) < 1e-16:
                    break
        return total if on is None else torch.where(on, total, psi)
    if kind == "add":
        half = n // 2
        low = (1 << half) - 1
        b = n - half
        target = (index & ~(low << b)) | ((((index >> b) + (index & low)) & low) << b)
        return torch.zeros_like(psi).index_copy_(0, target, psi)
    N, a = _modulus(case, seed)
    low = (1 << case["bits"]) - 1
    for k in range(n - case["bits"]):
        value = index & low
        moved = (index & ~low) | (value * pow(a, 1 << k, N) % N)
        target = torch.where((index >> (case["bits"] + k)) & 1 == 1, moved, index)
        # residues move to residues one to one; the rest of the register holds zeros
        held = (value < N).nonzero().reshape(-1)
        psi = torch.zeros_like(psi).index_copy_(0, target[held], psi[held])
    return psi
