"""A numpy interpreter of the records of blocking.compile_program (layouts,
scaled rotations, two-qubit gates in registers), for the tests on the CPU.
Factors are held as the kernels hold them: a LANE_PHASE multiplies the lane's
pending factor, which reaches the amplitudes at the next change of layout,
DENSE_LDS or store, so a range that the kernels leave is left here too."""

import numpy as np

from qibo_amd import blocking

LAYOUT0 = 0xBA9876543210
PAIRS = [(1, 0), (2, 0), (3, 0), (2, 1), (3, 1), (3, 2)]


def records(program, count, itemsize):
    cdt = np.complex128 if itemsize == 16 else np.complex64
    out, off = [], 0
    for _ in range(count):
        op, arg, nt, rreq = (int(x) for x in program[off: off + 4])
        nent = int.from_bytes(program[off + 4: off + 8], "little")
        raw = program[off + 8: off + 32]
        mat = np.frombuffer(program, dtype=cdt, count=nent, offset=off + 32)
        out.append((op, arg, nt, rreq, raw, mat))
        off += blocking.record_bytes(nent, itemsize)
    assert off == len(program)
    return out


def _nibbles(word):
    lay = [(word >> (4 * p)) & 15 for p in range(12)]
    assert sorted(lay) == list(range(12)) and word < 1 << 48
    return lay


def run_program(state, n, tile_bits, program, count, low):
    """Apply one compiled pass to a numpy state."""
    itemsize = state.dtype.itemsize
    rdt = np.float64 if itemsize == 16 else np.float32
    others = [b for b in range(n) if b not in tile_bits]
    base = np.zeros(2 ** len(others), dtype=np.int64)
    for i, b in enumerate(others):
        base |= ((np.arange(base.size) >> i) & 1) << b
    pos = np.arange(4096)

    def index(lay):  # global index of (tile, position)
        g = np.zeros(4096, dtype=np.int64)
        for p in range(12):
            g |= ((pos >> p) & 1) << tile_bits[lay[p]]
        return base[:, None] | g[None, :]

    recs = records(program, count, itemsize)
    assert recs[0][0] == blocking.OP_MAP and recs[0][1] == blocking.MAP_START
    lay = _nibbles(int.from_bytes(recs[0][4][:8], "little"))
    names = list(lay)  # as the kernel sees it; `lay` may run ahead between renames
    assert not set(lay[8:]) & set(range(low))
    gidx = index(lay)
    v = state[gidx].copy()
    pend = np.ones_like(v)
    lane = np.ones_like(v)  # the pending factor of LANE_PHASE records: the same on all registers of a lane
    qbit = None
    for op, arg, nt, rreq, raw, mat in recs[1:]:
        cmask = int.from_bytes(raw[:8], "little")
        bits = list(raw[8:16])
        tmask = int.from_bytes(raw[16:24], "little")
        gidx = index(names)
        reg = pos >> 8
        active = ((gidx & tmask) == tmask) if op != blocking.OP_ROTS and op != blocking.OP_ROT else None
        assert not any((tmask >> b) & 1 for b in tile_bits)
        if op == blocking.OP_MAP:
            assert qbit is None or arg == blocking.MAP_RELABEL
            if arg == blocking.MAP_RELABEL:
                names = _nibbles(cmask)
                continue
            assert arg == blocking.MAP_LAYOUT
            v, lane = v * lane, np.ones_like(v)
            frm, to = _nibbles(int.from_bytes(raw[8:16], "little")), _nibbles(cmask)
            full = np.empty_like(v)

            def local(lay):
                u = np.zeros(4096, dtype=np.int64)
                for p in range(12):
                    u |= ((pos >> p) & 1) << lay[p]
                return u
            full[:, local(frm)] = v
            v = full[:, local(to)]
            names = to
            continue
        if op == blocking.OP_DENSE_LDS:
            k = arg
            v, lane = v * lane, np.ones_like(v)
            tb = [tile_bits[b] for b in bits[:k]]
            assert sorted(bits[:k]) == bits[4: 4 + k]
            full = state.copy()
            full[gidx] = v
            sel = (np.arange(2**n) & (cmask | tmask)) == (cmask | tmask)
            zero = np.arange(2**n)[sel]
            for b in tb:
                zero = zero[((zero >> b) & 1) == 0]
            off = [sum(((r >> (k - 1 - t)) & 1) << tb[t] for t in range(k)) for r in range(2**k)]
            x = np.stack([full[zero | o] for o in off])
            y = mat.reshape(2**k, 2**k) @ x
            for r, o in enumerate(off):
                full[zero | o] = y[r]
            v = full[gidx]
            continue
        cond = np.ones_like(gidx, dtype=bool)
        if op not in (blocking.OP_ROT, blocking.OP_ROTS):
            cond = active & ((gidx & cmask) == cmask) & ((reg & rreq) == rreq)[None, :]
            regbits = sum(1 << tile_bits[names[8 + j]] for j in range(4))
            assert cmask & regbits == 0
        if qbit is not None and op in (blocking.OP_ROT, blocking.OP_ROTS, blocking.OP_DENSE1, blocking.OP_DENSE1_REAL,
                                       blocking.OP_FLIP):
            assert arg & 3 != qbit
        if qbit is not None and op == blocking.OP_DENSE2:
            assert qbit not in PAIRS[arg & 7]

        def pairs(j):
            i0 = pos[((pos >> (8 + j)) & 1) == 0]
            return i0, i0 | (1 << (8 + j))

        if op in (blocking.OP_ROT, blocking.OP_ROTS):
            i0, i1 = pairs(arg & 3)
            t = np.frombuffer(raw[:8], dtype=rdt)[0]
            s = np.frombuffer(raw[8:16], dtype=rdt)[0]
            if op == blocking.OP_ROTS:
                c, s = rdt(1), t
            else:
                assert abs(t) <= 1
                c = rdt(1) - t * s
            m = {0: [[c, -s], [s, c]], 1: [[c, s], [s, -c]], 2: [[c, -1j * s], [-1j * s, c]]}[arg >> 2]
            a, b = v[:, i0].copy(), v[:, i1].copy()
            v[:, i0], v[:, i1] = m[0][0] * a + m[0][1] * b, m[1][0] * a + m[1][1] * b
        elif op in (blocking.OP_DENSE1, blocking.OP_DENSE1_REAL, blocking.OP_FLIP):
            i0, i1 = pairs(arg & 3)
            m = [0, 1, 1, 0] if op == blocking.OP_FLIP else mat
            assert not (rreq >> (arg & 3)) & 1
            a, b = v[:, i0].copy(), v[:, i1].copy()
            ok = cond[:, i0]
            v[:, i0], v[:, i1] = np.where(ok, m[0] * a + m[1] * b, a), np.where(ok, m[2] * a + m[3] * b, b)
        elif op == blocking.OP_DENSE2:
            hi, lo = PAIRS[arg & 7]
            z = pos[(((pos >> (8 + hi)) & 1) == 0) & (((pos >> (8 + lo)) & 1) == 0)]
            at = [z, z | 1 << (8 + lo), z | 1 << (8 + hi), z | 1 << (8 + hi) | 1 << (8 + lo)]
            m = mat.reshape(4, 4)
            kind = arg >> 3
            keep = np.eye(4, dtype=bool) | np.eye(4, dtype=bool)[::-1] if kind >= 2 else np.ones((4, 4), dtype=bool)
            assert not np.any(m[~keep]) and (kind % 2 == 0 or not np.any(m.imag))
            x = [v[:, i].copy() for i in at]
            for r in range(4):
                v[:, at[r]] = sum(m[r, c] * x[c] for c in range(4) if keep[r, c])
        elif op == blocking.OP_REG_PHASE:
            assert cmask == 0 and rreq == 0 and tmask == 0
            dep = arg & 15
            assert all(mat[r] == 1 for r in range(16) if dep and not r & dep)
            v = v * mat[reg][None, :]
        elif op == blocking.OP_NEG:
            v = np.where(cond, -v, v)
        elif op in (blocking.OP_LANE_PHASE, blocking.OP_DIAG):
            di = np.zeros_like(gidx)
            for tb in bits[:nt]:
                if tb & blocking.REG_FLAG:
                    assert op == blocking.OP_DIAG
                    di = (di << 1) | ((pos >> (8 + (tb & 3))) & 1)[None, :]
                else:
                    assert tb not in [tile_bits[names[8 + j]] for j in range(4)]
                    di = (di << 1) | ((gidx >> tb) & 1)
            if op == blocking.OP_LANE_PHASE:
                assert rreq == 0
                lane = np.where(cond, lane * mat[di], lane)
            else:
                v = np.where(cond, v * mat[di], v)
        elif op == blocking.OP_LANE_REGPHASE:
            assert rreq == 0 and qbit in (None, arg)
            qbit = arg
            pend = np.where(cond & ((reg >> arg) & 1)[None, :].astype(bool), pend * mat[0], pend)
        elif op == blocking.OP_LRPMANY:
            assert rreq == 0 and cmask == 0 and tmask == 0 and qbit in (None, arg) and 3 <= nt <= 48
            qbit = arg
            for k, b in enumerate(mat[nt:].tobytes()[:nt]):
                assert bool(b & 0x80) == ((b & 63) not in tile_bits)
                assert (b & 63) not in [tile_bits[names[8 + j]] for j in range(4)]
                on = (((gidx >> (b & 63)) & 1) == 1) & ((reg >> arg) & 1)[None, :].astype(bool)
                pend = np.where(on, pend * mat[k], pend)
        elif op == blocking.OP_QFLUSH:
            assert qbit == arg
            v, pend, qbit = v * pend, np.ones_like(v), None
        else:
            raise AssertionError(f"record {op}")
    assert qbit is None
    v = v * lane
    assert not set(names[8:]) & set(range(low)), "a low bit is stored from a register"
    out = state.copy()
    out[index(names)] = v
    return out
