"""Pauli sums through tiles (needs an MI355X): the sizes and term tables where
the tile kernel changes its route, against numpy in double precision.

Masks inside the lane bits, on register bits, across both and over the whole
register (too many flip bits for a tile), coefficients real and imaginary
(odd and even numbers of Y), many Z strings of every register pattern, more
terms and masks than one launch holds, registers below and just above one
tile. Bound: each term adds 2^n products of unit size in double precision
(complex64 amplitudes are widened first), so 1e-12 of the coefficients' sum
covers them; the product state is rounded to the state's type at the end."""

import numpy as np
import pytest
import torch

from qibo_amd import _lib

pytestmark = pytest.mark.gpu


def _apply(psi, n, xm, zm, ny, c):
    idx = np.arange(2**n, dtype=np.uint64)
    out = np.zeros(2**n, dtype=np.complex128)
    for x, z, y, k in zip(xm, zm, ny, c):
        j = idx ^ np.uint64(x)
        parity = j & np.uint64(z)
        for s in (32, 16, 8, 4, 2, 1):
            parity ^= parity >> np.uint64(s)
        out += k * 1j ** int(y) * np.where(parity & np.uint64(1), -1.0, 1.0) * psi[j]
    return out


def _tables(n, rng):
    """Strings with masks of every kind; ny = the number of Y, as the package builds them."""
    full = (1 << n) - 1
    xs = [0, 1, 1 << (n - 1), 3, full, full ^ 1, 1 << (n // 2)]
    xs += [(1 << b) & full for b in (5, 6, 7, 8, 9, 10, 11)] + [0x181 & full, 0xF00 & full, 0x0F0 & full]
    xs += [int(x) for x in rng.integers(0, full + 1, size=6)]
    xs = [x for x in xs if x <= full]
    xm, zm = [], []
    for x in xs:
        for z in [0, x, full] + [int(z) for z in rng.integers(0, full + 1, size=3)]:
            xm.append(x)
            zm.append(z)
    zs = rng.integers(0, full + 1, size=90)  # more diagonal terms than one launch takes
    xm += [0] * len(zs)
    zm += [int(z) for z in zs]
    # up to 35 terms on one mask: more than a group takes
    xm += [3 & full] * 35
    zm += [int(z) for z in rng.integers(0, full + 1, size=35)]
    ny = [bin(x & z).count("1") for x, z in zip(xm, zm)]
    return (np.array(xm, dtype=np.uint64), np.array(zm, dtype=np.uint64), np.array(ny, dtype=np.int32),
            rng.normal(size=len(xm)))


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [1, 2, 7, 11, 12, 13, 15])
def test_pauli_tables_by_tiles(request, n, dtype, rng):
    be = request.getfixturevalue("backend" if dtype == "complex128" else "backend64")
    lib = be.lib
    xm, zm, ny, c = _tables(n, rng)
    nb = 3
    psi = rng.normal(size=(nb, 2**n)) + 1j * rng.normal(size=(nb, 2**n))
    psi = (psi / np.linalg.norm(psi, axis=1)[:, None]).astype(dtype)
    want = [_apply(p.astype(np.complex128), n, xm, zm, ny, c) for p in psi]
    energy = [float(np.real(np.vdot(p.astype(np.complex128), w))) for p, w in zip(psi, want)]
    scale = float(np.sum(np.abs(c)))
    dev = torch.from_numpy(psi).cuda()
    for b in range(nb):
        got = float(be.expectation_pauli(dev[b].clone(), n, xm, zm, ny, c))
        assert abs(got - energy[b]) <= 1e-12 * scale
    ws = torch.empty(lib.qsim_apply_pauli_sum_batched_workspace(nb, len(c)), dtype=torch.uint8, device="cuda")
    out = torch.full_like(dev, float("nan"))
    es = torch.full((nb,), float("nan"), dtype=torch.float64, device="cuda")
    _lib.check(lib.qsim_apply_pauli_sum_batched(dev.data_ptr(), nb, n, be._dtype_code(dev), len(c), xm.ctypes.data,
                                                zm.ctypes.data, ny.ctypes.data, c.ctypes.data, out.data_ptr(),
                                                es.data_ptr(), ws.data_ptr(), ws.numel(), be._stream(dev)), lib)
    # complex64: rounded to the state's type at the end of each of the (few) launches
    tol = (1e-12 if dtype == "complex128" else 1e-6) * scale
    assert np.max(np.abs(out.cpu().numpy() - np.array(want))) <= tol
    assert np.max(np.abs(es.cpu().numpy() - np.array(energy))) <= 1e-12 * scale
    one = be.apply_pauli_sum(dev[0].clone(), n, xm, zm, ny, c).cpu().numpy()
    assert np.max(np.abs(one - want[0])) <= tol


def _one_launch(kind, n, rng):
    """At most 64 terms: distinct X masks, diagonal terms, both, and terms of
    one mask with even and odd numbers of Y (an item each)."""
    full = (1 << n) - 1
    masks = [int(x) for x in rng.choice(np.arange(1, full), 64, replace=False)]
    xm = {"masks": masks, "diagonal": [0] * 64, "both": [0] * 32 + masks[:32], "more_diagonal": [0] * 48 + masks[:16],
          "parities": [m for m in masks[:32] for _ in range(2)], "one_mask": [5] * 64,
          "singles_then_one_mask": sorted(masks)[:48] + [full] * 16}[kind]
    zm = [int(z) for z in rng.integers(0, full + 1, size=len(xm))]
    if kind == "parities":  # the number of common bits even, then odd
        zm = [z ^ ((bin(x & z).count("1") + i) % 2) * (x & -x) for i, (x, z) in enumerate(zip(xm, zm))]
    ny = [bin(x & z).count("1") for x, z in zip(xm, zm)]
    return (np.array(xm, dtype=np.uint64), np.array(zm, dtype=np.uint64), np.array(ny, dtype=np.int32),
            rng.normal(size=len(xm)))


@pytest.mark.parametrize("n", [12, 20])
@pytest.mark.parametrize("kind", ["masks", "diagonal", "both", "more_diagonal", "parities", "one_mask",
                                  "singles_then_one_mask"])
def test_complex64_products_of_64_terms_round_once(backend64, kind, n, rng):
    """Sums of up to 64 terms are formed in double precision and rounded to
    complex64 once: half a unit in the last place of each component, 2^-24 of
    it, beside the 1e-13 of double-precision sums of 64 terms."""
    be, lib = backend64, backend64.lib
    xm, zm, ny, c = _one_launch(kind, n, rng)
    nb = 2 if n < 20 else 1
    psi = rng.normal(size=(nb, 2**n)) + 1j * rng.normal(size=(nb, 2**n))
    psi = (psi / np.linalg.norm(psi, axis=1)[:, None]).astype(np.complex64)
    want = np.array([_apply(p.astype(np.complex128), n, xm, zm, ny, c) for p in psi])
    dev = torch.from_numpy(psi).cuda()
    ws = torch.empty(lib.qsim_apply_pauli_sum_batched_workspace(nb, len(c)), dtype=torch.uint8, device="cuda")
    out, es = torch.empty_like(dev), torch.empty(nb, dtype=torch.float64, device="cuda")
    _lib.check(lib.qsim_apply_pauli_sum_batched(dev.data_ptr(), nb, n, be._dtype_code(dev), len(c), xm.ctypes.data,
                                                zm.ctypes.data, ny.ctypes.data, c.ctypes.data, out.data_ptr(),
                                                es.data_ptr(), ws.data_ptr(), ws.numel(), be._stream(dev)), lib)
    one = be.apply_pauli_sum(dev[0].clone(), n, xm, zm, ny, c).cpu().numpy()
    scale = float(np.sum(np.abs(c)))
    for b in range(nb):
        energy = float(np.real(np.vdot(psi[b].astype(np.complex128), want[b])))
        assert abs(float(es[b]) - energy) <= 1e-12 * scale
        assert abs(float(be.expectation_pauli(dev[b].clone(), n, xm, zm, ny, c)) - energy) <= 1e-12 * scale
    slack = 1e-13 * scale * float(np.max(np.abs(psi)))
    for got, ref in [(out.cpu().numpy(), want), (one, want[0])]:
        for part in ("real", "imag"):
            g, w = getattr(got, part).astype(np.float64), getattr(ref, part)
            assert np.all(np.abs(g - w) <= 2.0**-24 * np.abs(w) + slack)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [20, 22, 24])
def test_products_on_both_sides_of_the_rule(request, n, dtype, rng):
    """One state from 20 qubits on is multiplied term by term where the terms
    are few or leave the tile, else by tiles: the same product either way (to a
    unit in the last place of complex64, 1e-13 of the coefficients' sum)."""
    be = request.getfixturevalue("backend" if dtype == "complex128" else "backend64")
    psi = torch.randn(2**n, dtype=torch.complex128, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    psi = (psi / psi.norm()).to(getattr(torch, dtype))
    wide = psi.to(torch.complex128)
    high, idx = n - 1, torch.arange(2**n, device="cuda")
    for xm in ([1], [1 << high], [0] * 3 + [1 << high], [0, 0, 1, 2, 4, 8] * 4, [1 << high] * 6 + [3],
               [1 << b for b in range(n)] + [0] * 6):
        zm = [int(z) for z in rng.integers(0, 2**n, size=len(xm))]
        ny = [bin(x & z).count("1") for x, z in zip(xm, zm)]
        c = rng.normal(size=len(xm))
        want = torch.zeros_like(wide)
        for x, z, y, k in zip(xm, zm, ny, c):
            j = idx ^ x
            p = j & z
            for s in (32, 16, 8, 4, 2, 1):
                p = p ^ (p >> s)
            want += 1j**y * (float(k) * (1 - 2 * (p & 1)).to(torch.float64)) * wide[j]
        got = be.apply_pauli_sum(psi, n, np.array(xm, dtype=np.uint64), np.array(zm, dtype=np.uint64),
                                 np.array(ny, dtype=np.int32), c).to(torch.complex128)
        slack = 1e-13 * float(np.sum(np.abs(c))) * float(wide.abs().max())
        last = 2.0**-24 if dtype == "complex64" else 0.0
        err, ref = torch.view_as_real(got - want).abs(), torch.view_as_real(want).abs()
        assert bool((err <= last * ref + slack).all())


def test_batched_pauli_sum_refuses_bad_arguments(backend):
    lib = backend.lib
    n, nb = 5, 2
    x = np.zeros(1, dtype=np.uint64)
    y = np.zeros(1, dtype=np.int32)
    c = np.ones(1)
    psi = torch.zeros(nb, 2**n, dtype=torch.complex128, device="cuda")
    out, es = torch.empty_like(psi), torch.zeros(nb, dtype=torch.float64, device="cuda")
    need = lib.qsim_apply_pauli_sum_batched_workspace(nb, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")

    def call(nbatch=nb, out_ptr=out.data_ptr(), wsb=need, mask=x):
        return lib.qsim_apply_pauli_sum_batched(psi.data_ptr(), nbatch, n, _lib.C128, 1, mask.ctypes.data,
                                                x.ctypes.data, y.ctypes.data, c.ctypes.data, out_ptr, es.data_ptr(),
                                                ws.data_ptr(), wsb, backend._stream(psi))

    assert call() == _lib.OK
    assert call(nbatch=0) == _lib.EINVAL
    assert call(out_ptr=psi.data_ptr()) == _lib.EINVAL
    assert call(wsb=need - 1) == _lib.EINVAL
    assert call(mask=np.array([1 << n], dtype=np.uint64)) == _lib.EINVAL
