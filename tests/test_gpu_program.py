"""The programs the backend runs on the GPU (needs an MI355X): kernels
specialised to their records against the interpreter bit for bit, and the
final states against the numpy interpreter of the records and the oracle --
from a given state and from |0...0>, in both precisions, with every record
form (layouts, renames, scaled rotations, 4x4s in registers, flips)."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import OracleBackend
from qibo_amd import Circuit, _lib, blocking, gates, models
from qibo_amd.backend import GatePlanner, MI355XBackend, _dm_pair, _Op
from qibo_amd.serving import GPUExecutor, Request

from tests.program_records import records, run_program
from tests.specialize_programs import STEEP, mixed_circuit, steep_circuit
from tests.test_program import _phases, _random_state, _two_qubit

pytestmark = pytest.mark.gpu

ALL = (1 << 64) - 1


def _passes(circuit, n, cdt, low):
    planner = GatePlanner("complex128" if cdt == np.complex128 else "complex64")
    ops = [op for g in circuit.queue for op in planner.plan_ops(g)]
    for kind, payload in blocking.partition(iter(ops), n, low, False):
        if kind == "block":
            yield (payload[0],) + blocking.compile_program(payload[0], payload[1], n, cdt, low)


@pytest.mark.parametrize("cdt,tol", [(np.complex128, 1e-14), (np.complex64, 3e-6)])
def test_passes_interpreted_and_specialised(backend, rng, cdt, tol):
    lib = backend.lib
    n, code, low = 14, (_lib.C128 if cdt == np.complex128 else _lib.C64), (3 if cdt == np.complex128 else 4)
    isz = np.dtype(cdt).itemsize
    cases = [p for c in (mixed_circuit(n, rng, 1), _phases(n, rng), _two_qubit(n, rng), models.QFT(n))
             for p in list(_passes(c, n, cdt, low))[:3]]
    seen = set()
    for i, (bits, prog, count) in enumerate(cases):
        seen |= {r[0] for r in records(prog, count, isz)}
        dev = torch.from_numpy(np.frombuffer(prog + bytes(blocking.PAD_BYTES), dtype=np.uint8).copy()).cuda()
        tba = _lib.int_array(bits)
        handle = ctypes.c_uint64(0)
        for zero in (False, True):
            psi = _random_state(n, rng, cdt)
            start = torch.from_numpy(psi).cuda()
            a, b = start.clone(), start.clone()
            launch = lib.qsim_apply_blocked_from_zero if zero else lib.qsim_apply_blocked
            _lib.check(launch(a.data_ptr(), n, code, tba, dev.data_ptr(), len(prog), count, None), lib)
            if zero:
                psi = np.zeros_like(psi)
                psi[0] = 1
            held = next(k for k in range(13) if k == 12 or bits[k] != k)
            want = run_program(psi, n, list(bits), prog, count, max(3, min(held, low)))
            assert np.max(np.abs(a.cpu().numpy() - want)) < tol, (i, zero)
            rc = lib.qsim_blocked_specialize(prog, len(prog), count, code, int(zero), ctypes.byref(handle))
            if rc != 0:  # over the compile budget
                continue
            _lib.check(lib.qsim_apply_blocked_specialized(handle.value, b.data_ptr(), 1, n, code, tba, ALL,
                                                          dev.data_ptr(), 0, len(prog), count, None), lib)
            assert torch.equal(a, b), (i, zero)
    assert {1, 2, 5, 6, 7, 11, 12, 13, 14, 15, 16} <= seen


@pytest.mark.parametrize("specialize", [False, True])
@pytest.mark.parametrize("dtype,tol", [("complex128", 1e-12), ("complex64", 2e-5)])
@pytest.mark.parametrize("n", [5, 13, 16])
def test_circuits_match_the_oracle(n, dtype, tol, specialize, rng):
    be = MI355XBackend(dtype=dtype)
    be.specialize, be.specialize_after = specialize, 1
    circuits = [_phases(n, rng), _two_qubit(n, rng), models.QFT(n), models.random_layered_circuit(n, 8, 3, False)]
    for c in circuits[: 2 if specialize and n < 16 else 4]:
        want = OracleBackend().execute(c)
        for _ in range(2):
            got = be.execute_circuit(c).state().cpu().numpy()
            assert np.max(np.abs(got - want)) < tol
            be.wait_specializations()


@pytest.mark.parametrize("specialize", [False, True])
@pytest.mark.parametrize("dtype,tol", [("complex128", 1e-12), ("complex64", 2e-5)])
@pytest.mark.parametrize("n", [5, 12, 16])
def test_steep_rotations_beside_lane_phases(n, dtype, tol, specialize):
    """Pulses and phases whose cosines must not gather in the lanes' pending
    factor, as state vectors and (up to 6 qubits) density matrices."""
    be = MI355XBackend(dtype=dtype)
    be.specialize, be.specialize_after = specialize, 1
    for angle, repeats in STEEP:
        want = OracleBackend().execute(steep_circuit(n, angle, min(repeats, 30)))
        c = steep_circuit(n, angle, min(repeats, 30))
        for _ in range(2):
            got = be.execute_circuit(c).state().cpu().numpy()
            assert np.max(np.abs(got - want)) < tol
            be.wait_specializations()
        if n <= 6 and not specialize:
            got = be.execute_circuit(steep_circuit(n, angle, min(repeats, 30), density_matrix=True)).state().cpu().numpy()
            assert np.max(np.abs(got - np.outer(want, want.conj()))) < 2 * tol


@pytest.mark.parametrize("specialize", [False, True])
def test_swaps_alone_are_stored_after_every_load(specialize, rng):
    """A pass of renames only permutes its tiles in place without an exchange
    through LDS: no lane may store before the others have loaded."""
    n = 21
    be = MI355XBackend()
    be.specialize, be.specialize_after = specialize, 1
    c = Circuit(n)
    for q in range(9):
        c.add(gates.SWAP(q, 17 - q))
    host = _random_state(n, rng, np.complex128)
    at = np.arange(2**n)
    src = at & 7  # qubits 18-20 stay
    for q in range(18):
        src |= ((at >> (n - 1 - q)) & 1) << (n - 1 - (17 - q))
    psi, want = torch.from_numpy(host).cuda(), torch.from_numpy(host[src]).cuda()
    for _ in range(6):
        assert torch.equal(be.execute_circuit(c, initial_state=psi).state(), want)
        be.wait_specializations()


def _compile_pass_state(lib, ops, n):
    """|0...0> through compile_pass's records, registers below a tile as its low end."""
    pad = max(0, 12 - n)
    ops = [_Op(op.kind, tuple(q + pad for q in op.targets), tuple(q + pad for q in op.controls), op.data) for op in ops]
    state = torch.zeros(2 ** (n + pad), dtype=torch.complex64, device="cuda")
    state[0] = 1
    for kind, payload in blocking.partition(iter(ops), n + pad, 4, False):
        bits, pops = payload
        prog, count, _ = blocking.compile_pass(bits, pops, n + pad, np.complex64)
        dev = torch.from_numpy(np.frombuffer(prog + bytes(blocking.PAD_BYTES), dtype=np.uint8).copy()).cuda()
        _lib.check(lib.qsim_apply_blocked(state.data_ptr(), n + pad, _lib.C64, _lib.int_array(bits),
                                          dev.data_ptr(), len(prog), count, None), lib)
        torch.cuda.synchronize()
    return state[: 2**n]


@pytest.mark.parametrize("n", [5, 11, 12, 16, 18, 19])
def test_sampled_complex64_keeps_its_rounding(backend64, n):
    """complex64 registers keep compile_pass's records when shots are drawn
    (their rounding decides the seeded shots), whatever their size; the same
    circuit without a measurement runs compile_program's."""
    c = models.random_layered_circuit(n, 5, seed=4)
    planner = GatePlanner("complex64")
    ops = [op for g in c.queue if g.__class__.__name__ != "M" for op in planner.plan_ops(g)]
    state = _compile_pass_state(backend64.lib, ops, n)
    start = torch.zeros_like(state)
    start[0] = 1
    for _ in range(2):  # (compiled, then replayed)
        assert torch.equal(backend64.execute_circuit(c, initial_state=start).state(), state)
    backend64.set_seed(5)
    shots = backend64.execute_circuit(c, nshots=2000).samples()
    backend64.set_seed(5)
    want = backend64.sample_shots(backend64.calculate_probabilities(state, list(range(n)), n), 2000)
    got = (torch.as_tensor(shots).cpu().long() << torch.arange(n - 1, -1, -1)).sum(1)
    assert torch.equal(got, torch.as_tensor(want).cpu().long())
    plain = models.random_layered_circuit(n, 5, seed=4, measure=False)
    assert not torch.equal(backend64.execute_circuit(plain, initial_state=start).state(), state)


@pytest.mark.parametrize("density", [False, True])
def test_sampling_is_known_without_a_walk_over_the_queue(backend64, density, monkeypatch):
    """A complex64 circuit knows whether it is measured; looking through the
    queue of 300 gates on every call took 18 us."""
    asked = []
    keeps = MI355XBackend._keeps_samples
    monkeypatch.setattr(backend64, "_keeps_samples", lambda *a: asked.append(a[2]) or keeps(*a))
    for measure in (False, True):
        c = Circuit(6 if density else 13, density_matrix=density)
        for g in models.random_layered_circuit(c.nqubits, 2, seed=1, measure=measure).queue:
            c.add(g)
        for _ in range(2):
            backend64.execute_circuit(c)
            assert asked.pop() is measure and not asked


@pytest.mark.parametrize("cached", [True, False])
def test_sampled_complex64_density_matrices(cached):
    n = 7
    c = Circuit(n, density_matrix=True)
    for g in models.random_layered_circuit(n, 3, seed=4).queue:
        c.add(g)
    planner = GatePlanner("complex64")
    ops = [op for g in c.queue if g.__class__.__name__ != "M" for op in _dm_pair(planner.plan_gate(g), n)]
    be = MI355XBackend(dtype="complex64")
    be.program_cache = cached
    want = _compile_pass_state(be.lib, ops, 2 * n).view(2**n, 2**n)
    assert torch.equal(be.execute_circuit(c).state(), want)


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("n", [6, 13])
def test_sampled_complex64_served(backend64, n, small):
    """A served request for shots draws them from the state of a sampled run."""
    c = models.random_layered_circuit(n, 5, seed=9, measure=False)
    planner = GatePlanner("complex64")
    state = _compile_pass_state(backend64.lib, [op for g in c.queue for op in planner.plan_ops(g)], n)
    np.random.seed(3)
    want = backend64.sample_shots(backend64.calculate_probabilities(state, list(range(n)), n), 5000).cpu().numpy()
    executor = GPUExecutor({"complex64": backend64}, nstreams=2, batch_small=small)
    h = executor.start(Request(0, c, "complex64", "shots", 5000, seed=3))
    while not executor.done(h):
        executor.idle()
    np.testing.assert_array_equal(executor.result(h), want)
