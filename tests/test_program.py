"""The programs the backend runs (qsim_compile_program) on the CPU: a numpy
interpreter of their records must reproduce the oracle's gate-by-gate state,
over every gate family, orders and controls in and outside the tile, registers
of one tile and more, in both precisions; rotations by angles whose cosines
are tiny or zero keep the state in range; the same structure with other angles
gives the same records. A planted wrong pair order fails.

Bounds: a pass rounds each amplitude a few times per gate, so 1e-13 in
complex128 (states of norm 1, at most a few hundred gates) and 2e-5 in
complex64, whose matrices are rounded to 6e-8 first."""

import numpy as np
import pytest

from oracle import OracleBackend
from qibo_amd import Circuit, blocking, gates, models
from qibo_amd.backend import GatePlanner, _dm_pair, plan_matrix

from tests.program_records import PAIRS, records, run_program
from tests.specialize_programs import STEEP, mixed_circuit, steep_circuit


def _compiled(ops, n, cdt, low):
    for kind, payload in blocking.partition(iter(ops), n, low, False):
        if kind == "single":
            yield kind, payload, None, None
        else:
            bits, pops = payload
            prog, count = blocking.compile_program(bits, pops, n, cdt, low)
            yield kind, bits, prog, count


def _run(circuit, n, cdt, state, low=None):
    planner = GatePlanner("complex128" if cdt == np.complex128 else "complex64")
    ops = [op for g in circuit.queue for op in planner.plan_ops(g)]
    low = (3 if cdt == np.complex128 else 4) if low is None else low
    kinds = set()
    for kind, what, prog, count in _compiled(ops, n, cdt, low):
        if kind == "single":
            m = np.asarray(what.data, dtype=np.complex128)
            if what.kind == "diag":
                m = np.diag(m)
            elif what.kind == "swap":
                m = np.eye(4)[[0, 2, 1, 3]]
            state = _dense(state, n, m, what.targets, what.controls)
            continue
        held = 0
        while held < 12 and held < low and what[held] == held:
            held += 1
        state = run_program(state, n, list(what), prog, count, max(3, held))
        kinds |= {(r[0], r[1] if r[0] in (blocking.OP_MAP, blocking.OP_DENSE2) else 0)
                  for r in records(prog, count, state.dtype.itemsize)}
    return state, kinds


def _dense(state, n, m, targets, controls):
    t = state.reshape((2,) * n).copy()
    sel = tuple(1 if q in controls else slice(None) for q in range(n))
    sub = t[sel]
    left = [q for q in range(n) if q not in controls]
    axes = [left.index(q) for q in targets]
    k = len(axes)
    y = np.tensordot(m.reshape((2,) * (2 * k)), sub, axes=(range(k, 2 * k), axes))
    t[sel] = np.moveaxis(y, range(k), axes)
    return t.reshape(-1).astype(state.dtype)


def _oracle(circuit, n, state):
    ob = OracleBackend()
    state = state.astype(np.complex128)
    for g in circuit.queue:
        state = ob.apply_gate(g, state, n)
    return state


def _random_state(n, rng, cdt):
    psi = rng.normal(size=2**n) + 1j * rng.normal(size=2**n)
    return (psi / np.linalg.norm(psi)).astype(cdt)


def _phases(n, rng):
    """Diagonal gates between every kind of bits, between rotations."""
    c = Circuit(n)
    for _ in range(2):
        for q in range(n):
            c.add(gates.RX(q, float(rng.uniform(-6, 6))))
        for _ in range(2 * n):
            a, b, d = (int(x) for x in rng.choice(n, 3, replace=False))
            c.add(gates.RZZ(a, b, float(rng.uniform(-6, 6))))
            c.add(gates.CRZ(b, d, float(rng.uniform(-6, 6))))
            c.add(gates.CU1(a, d, float(rng.uniform(-6, 6))))
            c.add(gates.RZ(b, float(rng.uniform(-6, 6))).controlled_by(a, d))
    return c


def _two_qubit(n, rng):
    c = Circuit(n)
    for _ in range(30):
        a, b, d = (int(x) for x in rng.choice(n, 3, replace=False))
        c.add(gates.iSWAP(a, b))
        c.add(gates.SWAP(b, d))
        c.add(gates.RXX(a, d, float(rng.uniform(-6, 6))))
        c.add(gates.fSim(d, b, float(rng.uniform(-6, 6)), 0.7))
        c.add(gates.CNOT(a, b))
        c.add(gates.H(a))
        c.add(gates.SWAP(a, d).controlled_by(b))
        c.add(gates.FSWAP(d, a))
        c.add(gates.Unitary(np.linalg.qr(rng.normal(size=(4, 4)))[0], b, a))
    return c


@pytest.mark.parametrize("cdt,tol", [(np.complex128, 1e-13), (np.complex64, 2e-5)])
@pytest.mark.parametrize("family", ["mixed", "phases", "two_qubit", "layered", "qft", "ansatz"])
@pytest.mark.parametrize("n", [12, 13, 15])
def test_programs_match_the_oracle(family, n, cdt, tol, rng):
    make = {"mixed": lambda: mixed_circuit(n, rng, 2), "phases": lambda: _phases(n, rng),
            "two_qubit": lambda: _two_qubit(n, rng), "qft": lambda: models.QFT(n),
            "layered": lambda: models.random_layered_circuit(n, 6, seed=int(rng.integers(1000)), measure=False),
            "ansatz": lambda: models.hardware_efficient_ansatz(n, 2, rng.uniform(0, 6, 4 * n))}
    circuit = make[family]()
    psi = _random_state(n, rng, cdt)
    got, kinds = _run(circuit, n, cdt, psi)
    assert np.max(np.abs(got - _oracle(circuit, n, psi))) < tol
    if family in ("layered", "qft", "phases"):
        assert (blocking.OP_ROTS, 0) in kinds and (blocking.OP_ROT, 0) not in kinds
    if family == "two_qubit":
        assert {(blocking.OP_DENSE2, a) for a in range(32)} & kinds and (blocking.OP_FLIP, 0) in kinds


@pytest.mark.parametrize("low", [0, 2, 3, 4, 6])
def test_low_bits(low, rng):
    n = 14
    circuit = _two_qubit(n, rng)
    psi = _random_state(n, rng, np.complex128)
    got, _ = _run(circuit, n, np.complex128, psi, low)
    assert np.max(np.abs(got - _oracle(circuit, n, psi))) < 1e-13


@pytest.mark.parametrize("cdt,tol", [(np.complex128, 1e-13), (np.complex64, 2e-5)])
def test_steep_rotations(cdt, tol, rng):
    """Rotations by pi (cosine 6e-17, exactly zero or below the floor when
    multiplied), by small angles and near pi, many in a row with and without
    another record to take the cosines."""
    n = 12
    for tail in (True, False):
        circuit = Circuit(n)
        for k in range(4):
            for q in range(n):
                angle = [np.pi, np.pi - 1e-9, 1e-12, -np.pi, 3.0][(q + k) % 5]
                circuit.add((gates.RY if q % 2 else gates.RX)(q, float(angle)))
                circuit.add(gates.Unitary(np.array([[0.0, -1.0], [1.0, 0.0]]), q))
        if tail:
            for q in range(n):
                circuit.add(gates.RZ(q, 0.3 * q))
                circuit.add(gates.RY(q, 3.1))
        psi = _random_state(n, rng, cdt)
        got, _ = _run(circuit, n, cdt, psi)
        assert np.all(np.isfinite(got))
        assert np.max(np.abs(got - _oracle(circuit, n, psi))) < tol


@pytest.mark.parametrize("cdt,tol", [(np.complex128, 1e-13), (np.complex64, 2e-5)])
@pytest.mark.parametrize("angle,repeats", STEEP)
@pytest.mark.parametrize("n", [2, 5, 8, 12, 13, 16])
def test_steep_rotations_beside_lane_phases(n, angle, repeats, cdt, tol, rng):
    """Pulses on one qubit with phases on another between them: the phases wait
    in the lane's factor while the rotations run, so no cosine may wait there
    with them. From |0...0> and from a dense state; registers below a tile run
    as the low end of one."""
    if n > 13 and repeats > 30:
        repeats = 30  # (the interpreter's time)
    pad = max(0, 12 - n)
    circuit = steep_circuit(n, angle, repeats, pad)
    first = np.zeros(2 ** (n + pad), dtype=cdt)
    first[0] = 1
    second = np.zeros_like(first)
    second[: 2**n] = _random_state(n, rng, cdt)
    for psi in (first, second):
        got, _ = _run(circuit, n + pad, cdt, psi)
        assert np.all(np.isfinite(got))
        assert np.max(np.abs(got - _oracle(circuit, n + pad, psi))) < tol


@pytest.mark.parametrize("nrot", [1, 4, 5])
def test_rotations_alone(nrot, rng):
    """No record to take the cosines: shears, or one table for five and more."""
    circuit = Circuit(12)
    for q in range(nrot):
        circuit.add(gates.RY(q, 0.1 + q))
    psi = _random_state(12, rng, np.complex128)
    got, kinds = _run(circuit, 12, np.complex128, psi)
    assert np.max(np.abs(got - _oracle(circuit, 12, psi))) < 1e-15
    assert ((blocking.OP_ROTS, 0) in kinds) == (nrot >= 5)


def _rotations(n, layers, rng, kinds=("RX", "RY"), diagonals=1):
    """Layers of rotations with few diagonals between them."""
    c = Circuit(n)
    for layer in range(layers):
        for kind in kinds:
            for q in range(n):
                c.add(getattr(gates, kind)(q, float(rng.uniform(0, 2 * np.pi))))
        if layer < diagonals:
            c.add(gates.CZ(layer, layer + 1))
    return c


@pytest.mark.parametrize("cdt", [np.complex128, np.complex64])
@pytest.mark.parametrize("circuit", ["layered", "rotations12", "rotations14", "diagonals", "none"])
def test_other_angles_give_the_same_records(circuit, cdt):
    """Which rotations are scaled, and where tables are added for them, follows
    from the structure: kernels specialised to it serve every parameter set."""
    make = {"layered": lambda r: models.random_layered_circuit(15, 10, seed=int(r.integers(1000)), measure=False),
            "rotations12": lambda r: _rotations(12, 10, r), "rotations14": lambda r: _rotations(14, 20, r),
            "diagonals": lambda r: _rotations(13, 9, r, ("RX", "RY", "RZ"), 9),
            "none": lambda r: _rotations(12, 12, r, diagonals=0)}[circuit]
    low = 3 if cdt == np.complex128 else 4
    seqs, scaled, sheared = [], 0, 0
    for seed in range(10):
        planner = GatePlanner("complex128" if cdt == np.complex128 else "complex64")
        c = make(np.random.default_rng(seed))
        ops = [op for g in c.queue for op in planner.plan_ops(g)]
        seqs.append([[(r[0], r[1], len(r[5])) for r in records(prog, count, np.dtype(cdt).itemsize)]
                     for _, _, prog, count in _compiled(ops, c.nqubits, cdt, low)])
        scaled += sum(r[0] == blocking.OP_ROTS for s in seqs[-1] for r in s)
        sheared += sum(r[0] == blocking.OP_ROT for s in seqs[-1] for r in s)
    assert all(s == seqs[0] for s in seqs[1:])
    assert sheared <= 0.02 * scaled  # (the last few before a table that would not pay)


@pytest.mark.parametrize("cdt,tol", [(np.complex128, 1e-13), (np.complex64, 2e-5)])
@pytest.mark.parametrize("diagonals", [0, 1, 7])
def test_long_runs_of_rotations(diagonals, cdt, tol, rng):
    """Runs past the limit of one table, before and after the first record
    that takes cosines."""
    circuit = _rotations(13, 14, rng, diagonals=diagonals)
    psi = _random_state(13, rng, cdt)
    got, _ = _run(circuit, 13, cdt, psi)
    assert np.max(np.abs(got - _oracle(circuit, 13, psi))) < tol


def _extended(circuit, n, state):
    """RX, RZZ and CRZ circuits in extended precision, angles included."""
    state = state.astype(np.clongdouble)
    idx = np.arange(2**n)
    for g in circuit.queue:
        half = np.longdouble(g.parameters[0]) / 2
        c, s = np.cos(half), np.sin(half)
        bit = [(idx >> (n - 1 - q)) & 1 for q in g.qubits]
        if g.name == "rx":
            state = c * state - 1j * s * state[idx ^ (1 << (n - 1 - g.qubits[0]))]
        else:  # the sign of the phase: by parity, or by the target under the control
            sign = np.where(bit[0] ^ bit[1], 1, -1) if g.name == "rzz" else np.where(bit[0] == 1, 2 * bit[1] - 1, 0)
            state = np.where(sign == 0, 1, c + 1j * s * sign) * state
    return state


def test_phases_cost_no_precision():
    """Diagonal gates between register and lane bits, split into a table, a
    lane's phase and a controlled phase, together round an amplitude no more
    often than gate by gate: the error against extended precision is at most the
    oracle's, which rounds once per gate (with a tenth for their scatter over
    four circuits; entries of split gates rounded one by one gave 1.4 times)."""
    n, ours, oracle = 14, 0.0, 0.0
    for seed in range(4):
        rng = np.random.default_rng(seed)
        c = Circuit(n)
        for _ in range(8):
            for q in range(n):
                c.add(gates.RX(q, float(rng.uniform(0, 6))))
            for _ in range(n):
                for kind in (gates.CRZ, gates.RZZ):
                    a, b = (int(x) for x in rng.choice(n, 2, replace=False))
                    c.add(kind(a, b, float(rng.uniform(0, 6))))
        psi = _random_state(n, rng, np.complex128)
        want = _extended(c, n, psi)
        got, _ = _run(c, n, np.complex128, psi)
        ours += float(np.linalg.norm((got - want).astype(np.complex128)))
        oracle += float(np.linalg.norm((_oracle(c, n, psi) - want).astype(np.complex128)))
    assert ours <= 1.1 * oracle


@pytest.mark.parametrize("n,layers", [(12, 10), (12, 20), (14, 10), (20, 10)])
def test_layouts_change_no_more_often_than_mappings(n, layers):
    """The free choice of register bits is not behind compile_pass's three groups."""
    planner = GatePlanner()
    ops = [op for g in models.random_layered_circuit(n, layers, seed=3, measure=False).queue for op in planner.plan_ops(g)]
    free = fixed = 0
    for kind, payload in blocking.partition(iter(ops), n, 3, False):
        prog, count = blocking.compile_program(payload[0], payload[1], n, np.complex128, 3)
        free += sum(r[0] == blocking.OP_MAP and r[1] == blocking.MAP_LAYOUT for r in records(prog, count, 16))
        fixed += blocking.compile_pass(payload[0], payload[1], n, np.complex128)[2]
    assert free <= fixed + 1  # (the tile may be stored from the last layout only)


def test_density_ops(rng):
    """Conjugate pairs and real transfer matrices on (row, column) qubits run
    in registers (the channel's 4x4 touches the pairs (00, 11) and (01, 10))."""
    n = 7
    planner = GatePlanner()
    psi = _random_state(2 * n, rng, np.complex128)
    ops = []
    for q in range(n):
        ops.extend(_dm_pair(planner.plan_gate(gates.RY(q, 0.3 + q)), n))
        ops.append(plan_matrix(planner.channel_transfer_matrix(gates.DepolarizingChannel((q,), 0.1)), (q, q + n), ()))
        ops.append(plan_matrix(planner.channel_transfer_matrix(gates.AmplitudeDampingChannel(q, 0.2)), (q, q + n), ()))
    want = psi
    for op in ops:
        m = np.diag(op.data) if op.kind == "diag" else np.asarray(op.data)
        want = _dense(want, 2 * n, m, op.targets, op.controls)
    got, kinds = psi, set()
    for kind, bits, prog, count in _compiled(ops, 2 * n, np.complex128, 3):
        assert kind == "block"
        got = run_program(got, 2 * n, list(bits), prog, count, 3)
        kinds |= {(r[0], r[1] >> 3 if r[0] == blocking.OP_DENSE2 else 0) for r in records(prog, count, 16)}
    assert np.max(np.abs(got - want)) < 1e-13
    assert (blocking.OP_DENSE2, 3) in kinds and (blocking.OP_DENSE_LDS, 0) not in kinds


def test_a_wrong_pair_order_fails(rng, monkeypatch):
    monkeypatch.setattr("tests.program_records.PAIRS", [(lo, hi) for hi, lo in PAIRS])
    circuit = Circuit(12)
    circuit.add(gates.Unitary(np.linalg.qr(rng.normal(size=(4, 4)))[0], 9, 3))
    circuit.add(gates.RY(9, 0.4))
    psi = _random_state(12, rng, np.complex128)
    got, _ = _run(circuit, 12, np.complex128, psi)
    assert np.max(np.abs(got - _oracle(circuit, 12, psi))) > 1e-3
