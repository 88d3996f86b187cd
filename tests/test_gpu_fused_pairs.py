"""Two dense blocks in one pass against two passes, and the pairing of a circuit."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _unitary(rng, k):
    q, _ = np.linalg.qr(rng.normal(size=(2**k, 2**k)) + 1j * rng.normal(size=(2**k, 2**k)))
    return q


@pytest.mark.parametrize(
    "n,first,second",
    [
        (13, (0, 1, 2, 3, 4), (5, 6, 7, 8, 9)),  # one tile, no target among the low bits' lines
        (13, (12, 10, 9, 8, 7), (0, 6, 3, 9, 12)),  # reversed and overlapping targets
        (14, (13, 2, 7, 0), (1, 12, 5, 8, 3)),
        (15, (4, 9, 14, 1, 6), (0, 3, 10, 13)),
        (17, (16, 15, 14, 13), (0, 1, 2, 3)),
        (22, (0, 1, 2, 3, 4), (0, 1, 2, 3, 4)),  # more tiles than resident workgroups; the same targets
        (22, (3, 20, 9, 14, 7), (19, 1, 11, 5, 17)),
    ],
)
def test_pair_is_bitwise_two_blocks(backend, n, first, second):
    from qibo_amd import _lib

    rng = np.random.default_rng(n)
    psi = torch.from_numpy(rng.normal(size=2**n) + 1j * rng.normal(size=2**n)).cuda()
    mats = [torch.from_numpy(_unitary(rng, len(t))).cuda() for t in (first, second)]
    lib, two, one = backend.lib, psi.clone(), psi.clone()
    stream = torch.cuda.current_stream().cuda_stream
    for m, t in zip(mats, (first, second)):
        _lib.check(lib.qsim_apply_fused(two.data_ptr(), n, _lib.C128, _lib.int_array(t), len(t), m.data_ptr(), stream), lib)
    _lib.check(lib.qsim_apply_fused_pair(one.data_ptr(), None, n, _lib.C128, _lib.int_array(first), len(first),
                                         mats[0].data_ptr(), _lib.int_array(second), len(second), mats[1].data_ptr(),
                                         stream), lib)
    assert torch.equal(torch.view_as_real(one), torch.view_as_real(two))


def test_pair_refuses_what_it_does_not_cover(backend):
    from qibo_amd import _lib

    psi = torch.zeros(2**13, dtype=torch.complex128, device="cuda")
    m = torch.eye(32, dtype=torch.complex128, device="cuda")
    lib = backend.lib

    def call(n, code, t1, t2, source=None):
        return lib.qsim_apply_fused_pair(psi.data_ptr(), source, n, code, _lib.int_array(t1), len(t1), m.data_ptr(),
                                         _lib.int_array(t2), len(t2), m.data_ptr(), 0)

    five = (0, 1, 2, 3, 4)
    assert call(12, _lib.C128, five, five) != 0
    assert call(13, _lib.C64, five, five) != 0
    assert call(13, _lib.C128, five, (0, 1, 2)) != 0
    assert call(13, _lib.C128, (0, 1, 2, 3, 3), five) != 0
    assert call(13, _lib.C128, five, (0, 1, 2, 3, 13)) != 0
    assert call(13, _lib.C128, five, five, psi.data_ptr() + 4096) != 0  # overlaps the state


@pytest.mark.parametrize("count", [1, 2, 3, 5])
def test_circuit_of_blocks_and_gates(backend, count):
    """Blocks with gates between them: in order, from |0...0>, planned and replayed."""
    from qibo_amd import Circuit, gates

    n, rng = 13, np.random.default_rng(count)
    c = Circuit(n)
    for q in range(n):
        c.add(gates.RY(q, theta=0.1 + q))
    for i in range(count):
        qubits = tuple(int(q) for q in rng.permutation(n)[: 4 + i % 2])
        c.add(gates.Unitary(_unitary(rng, len(qubits)), *qubits, check_unitary=False))
        if i == 2:
            c.add(gates.CNOT(0, 5))
            c.add(gates.H(7))
    for _ in range(3):
        c._final_state = None
        got = backend.execute_circuit(c).state()
        got = torch.as_tensor(got).cuda()
        ref = backend.zero_state(n)
        for g in c.queue:
            ref = backend.apply_gate(g, ref, n)
        # each amplitude sums at most 32 products per block, unit vectors
        assert float((got - ref).abs().max()) < 32 * 2.3e-16 * (count + 2)
