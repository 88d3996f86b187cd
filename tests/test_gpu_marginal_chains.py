"""Marginals whose outcomes add long chains (needs an MI355X): the workgroup
kernel that adds from LDS, at the chain lengths and outcome counts where its
split changes, against numpy's own sum bit for bit. The cases cover the three
kinds of values (single probabilities, leaves of a short trailing run, run
sums), chains around the shortest it takes (2^7) and around one chunk, one to
64 outcomes per workgroup, several chunks, requested orders that are not
ascending, and run sums of every length (128 to several buffers of 8192)."""

import numpy as np
import pytest
import torch

from oracle import OracleBackend

pytestmark = pytest.mark.gpu

_CASES = [
    # last qubit measured: chains of 2^6, 2^7, 2^8 and 2^13; 1, 2, 8 and 64 outcomes per workgroup
    (9, [8, 0, 3]), (10, [9, 1, 2]), (9, [8]), (14, [13]), (16, [15, 14, 13]), (20, [int(q) for q in range(7, 20)]),
    (17, [16, 0, 9, 4, 2, 11, 14, 7, 1]), (21, list(range(20, 6, -1))), (16, [3, 15, 8]),
    # short trailing runs of 2, 8 and 64
    (13, [11, 2]), (16, [12, 0, 6]), (17, [10, 3]), (19, list(range(0, 10)) + [17]),
    # run sums of 128, 512, 1024, 2048, 8192 and several buffers, short and long chains of them
    (7, [0]), (8, [0]), (10, [1, 0]), (17, [9]), (16, [5, 2]), (15, [4]), (16, [3, 0]), (18, [4, 2]), (18, [0]), (20, [12]),
    (21, [1]),
]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n,qubits", _CASES)
def test_chains_bitwise(request, n, qubits, dtype, rng):
    backend = request.getfixturevalue("backend" if dtype == "complex128" else "backend64")
    # amplitudes over many orders of magnitude: an addition out of order shows
    psi = rng.normal(size=2**n) * np.exp(4 * rng.normal(size=2**n)) + 1j * rng.normal(size=2**n)
    psi = (psi / np.linalg.norm(psi)).astype(dtype)
    want = OracleBackend(dtype).calculate_probabilities(psi, qubits, n)
    got = backend.calculate_probabilities(torch.from_numpy(psi).cuda(), qubits, n).cpu().numpy()
    assert got.dtype == want.dtype
    assert np.array_equal(got, want), np.max(np.abs(got - want))
