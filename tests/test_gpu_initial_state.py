"""Circuits on an initial state that the first pass reads in place: the result
is bitwise that of a run on a copy, and the initial state stays as it was."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _circuit(kind, n):
    from qibo_amd import Circuit, gates, models

    rng = np.random.default_rng(n)
    c = Circuit(n)
    if kind in ("blocks", "block"):
        for i in range(2 if kind == "blocks" else 1):
            q, _ = np.linalg.qr(rng.normal(size=(32, 32)) + 1j * rng.normal(size=(32, 32)))
            c.add(gates.Unitary(q, *(int(x) for x in rng.permutation(n)[:5]), check_unitary=False))
    elif kind == "passes":
        return models.QFT(n)
    elif kind == "one":
        c.add(gates.CRX(0, n - 1, theta=0.3))
    return c


@pytest.mark.parametrize("kind", ["blocks", "block", "passes", "one", "empty"])
@pytest.mark.parametrize("n", [11, 12, 13, 18])
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_initial_state_is_read_in_place(kind, n, dtype, request):
    backend = request.getfixturevalue("backend" if dtype == "complex128" else "backend64")
    gen = torch.Generator().manual_seed(n)
    psi = torch.randn(2**n, dtype=torch.complex128, generator=gen).to(device="cuda", dtype=getattr(torch, dtype))
    before = psi.clone()
    for _ in range(3):  # planned, replayed, and with specialised kernels
        c = _circuit(kind, n)
        got = backend.execute_circuit(c, initial_state=psi).state()
        backend.wait_specializations()
        assert torch.equal(torch.view_as_real(psi), torch.view_as_real(before))
        assert torch.as_tensor(got).data_ptr() != psi.data_ptr()
        ref = backend.run_queue(_circuit(kind, n).queue, psi.clone(), n)
        assert torch.equal(torch.view_as_real(torch.as_tensor(got).to("cuda")), torch.view_as_real(ref))


def test_states_that_are_copied_first(backend):
    """Views, conjugates, other dtypes and host arrays: as before, through a copy."""
    n = 13
    psi = torch.randn(2**n, dtype=torch.complex128).cuda()
    c = _circuit("passes", n)
    run = lambda s: torch.as_tensor(backend.execute_circuit(_circuit("passes", n), initial_state=s).state()).cuda()  # noqa: E731
    ref = run(psi)
    assert torch.equal(run(psi.cpu().numpy()), ref)
    # a strided view
    twice = torch.zeros(2**n, 2, dtype=torch.complex128, device="cuda")
    twice[:, 0] = psi
    before = twice.clone()
    assert not twice[:, 0].is_contiguous() and torch.equal(run(twice[:, 0]), ref)
    assert torch.equal(twice, before)
    # a lazily conjugated one
    lazy = psi.conj()
    assert lazy.is_conj() and torch.equal(run(lazy), run(lazy.resolve_conj()))
    # one that autograd follows
    assert torch.equal(run(psi.clone().requires_grad_()).detach(), ref)
    single = psi.to(torch.complex64)
    assert torch.equal(run(single), run(single.to(torch.complex128)))
    with pytest.raises(ValueError):
        backend.execute_circuit(c, initial_state=psi[:-1])


def test_a_state_at_an_odd_address_is_copied_first(backend64):
    """complex64 views can start between the 16-byte lines that the passes read."""
    n = 13
    buf = torch.randn(2**n + 1, dtype=torch.complex64).cuda()
    psi = buf[1:]
    assert psi.data_ptr() % 16 == 8
    run = lambda s: backend64.execute_circuit(_circuit("passes", n), initial_state=s).state()  # noqa: E731
    before = buf.clone()
    assert torch.equal(run(psi), run(psi.clone()))
    assert torch.equal(buf, before)


def test_source_must_not_overlap(backend):
    from qibo_amd import _lib

    buf = torch.zeros(2**13 + 16, dtype=torch.complex128, device="cuda")
    bits = _lib.int_array(range(12))
    lib = backend.lib
    call = lambda s, f: lib.qsim_apply_blocked_from(s, f, 12, _lib.C128, bits, 0, 0, 0, 0)  # noqa: E731
    assert call(buf.data_ptr(), buf.data_ptr() + 16) != 0
    assert call(buf.data_ptr(), 0) != 0
    assert call(buf.data_ptr(), buf.data_ptr() + 16 * 2**12 + 8) != 0
    assert call(buf.data_ptr(), buf.data_ptr() + 16 * 2**12) == 0
