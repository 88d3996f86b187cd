// What the two record compilers share (host code): planned gates as they come
// over the C ABI, the record writer, the rotation forms of a 2x2.
#pragma once

#include <stdint.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "qsim_common.h"

namespace {

constexpr int kTileBits = 12;
constexpr int kHeader = 32;
constexpr int kDescInts = 44;  // kind, ntargets, ncontrols, -, targets[5], controls[35]
constexpr int kMaxTargets = 5;
constexpr int kMaxControls = 35;
constexpr int kRegGroups[3][4] = {{8, 9, 10, 11}, {4, 5, 6, 7}, {0, 1, 2, 3}};
constexpr uint32_t kRegFlag = 0x80;

enum Kind { kNoop = 0, kDiag = 1, kSwap = 2, kDense = 3 };
enum Rec : uint8_t {
  kRDiag = 0, kRDense1 = 1, kRMap = 2, kRDenseLds = 3, kRDense1Real = 4, kRRegPhase = 5, kRLanePhase = 6,
  kRNeg = 7, kRRot = 10, kRLaneRegPhase = 11, kRQFlush = 12
};

struct C {
  double re, im;
};

inline C cmulf(C a, C b) { return {std::fma(a.re, b.re, -(a.im * b.im)), std::fma(a.re, b.im, a.im * b.re)}; }
inline bool ceq(C a, C b) { return a.re == b.re && a.im == b.im; }

struct Op {
  int kind, nt, nc;
  int t[kMaxTargets];
  int c[kMaxControls];
  const C* data;
  int ndata;
  uint64_t nd_mask, all_mask;
};

struct Writer {
  uint8_t* out;
  size_t cap, len = 0;
  int itemsize;
  int count = 0;
  bool overflow = false;
  long absorb_off = -1;  // byte offset of the entries of the first unconditional linear record
  int absorb_n = 0;

  // Overwrite the n entries at byte offset `off` (complex128 values, stored in
  // the record's precision).
  void rewrite(long off, const C* data, int n) {
    uint8_t* e = out + off;
    for (int i = 0; i < n; ++i) {
      if (itemsize == 16) {
        std::memcpy(e + 16 * i, &data[i].re, 8);
        std::memcpy(e + 16 * i + 8, &data[i].im, 8);
      } else {
        const float re = float(data[i].re), im = float(data[i].im);
        std::memcpy(e + 8 * i, &re, 4);
        std::memcpy(e + 8 * i + 4, &im, 4);
      }
    }
  }

  void emit(uint8_t op, int arg, uint64_t cmask, int nt, const int* bits, int nbits, const C* data, int ndata,
            int rreq = 0) {
    const size_t raw = size_t(ndata) * size_t(itemsize);
    const size_t rec = kHeader + (raw + 15) / 16 * 16;
    if (len + rec > cap) {
      overflow = true;
      return;
    }
    if (absorb_off < 0 && cmask == 0 && rreq == 0 && data != nullptr &&
        (op == kRDense1 || op == kRDense1Real || op == kRRegPhase || op == kRLanePhase || op == kRDiag)) {
      absorb_off = long(len + kHeader);
      absorb_n = ndata;
    }
    uint8_t* h = out + len;
    std::memset(h, 0, rec);
    h[0] = op;
    h[1] = uint8_t(arg);
    h[2] = uint8_t(nt);
    h[3] = uint8_t(rreq);
    const uint32_t nent = uint32_t(ndata);
    std::memcpy(h + 4, &nent, 4);
    std::memcpy(h + 8, &cmask, 8);
    for (int i = 0; i < nbits && i < 8; ++i) h[16 + i] = uint8_t(bits[i]);
    uint8_t* e = h + kHeader;
    for (int i = 0; i < ndata; ++i) {
      if (itemsize == 16) {
        std::memcpy(e + 16 * i, &data[i].re, 8);
        std::memcpy(e + 16 * i + 8, &data[i].im, 8);
      } else {
        const float re = float(data[i].re), im = float(data[i].im);
        std::memcpy(e + 8 * i, &re, 4);
        std::memcpy(e + 8 * i + 4, &im, 4);
      }
    }
    len += rec;
    ++count;
  }

  // ROT record: no entries, (t, s) in the header's cmask and bits fields
  // (float64 at bytes 8 and 16; complex64: float32 at bytes 8 and 16)
  void emit_rot(int arg, double t, double s) {
    if (len + kHeader > cap) {
      overflow = true;
      return;
    }
    uint8_t* h = out + len;
    std::memset(h, 0, kHeader);
    h[0] = kRRot;
    h[1] = uint8_t(arg);
    if (itemsize == 16) {
      std::memcpy(h + 8, &t, 8);
      std::memcpy(h + 16, &s, 8);
    } else {
      const float tf = float(t), sf = float(s);
      std::memcpy(h + 8, &tf, 4);
      std::memcpy(h + 16, &sf, 4);
    }
    len += kHeader;
    ++count;
  }

  void negate_absorbed() {
    for (int i = 0; i < 2 * absorb_n; ++i) {
      uint8_t* p = out + absorb_off + size_t(i) * size_t(itemsize / 2);
      if (itemsize == 16) {
        double v;
        std::memcpy(&v, p, 8);
        v = -v;
        std::memcpy(p, &v, 8);
      } else {
        float v;
        std::memcpy(&v, p, 4);
        v = -v;
        std::memcpy(p, &v, 4);
      }
    }
  }
};

// (mode, t, s, negated) of a 2x2 of the ROT forms with |c^2 + s^2 - 1| <= tol
// (1e-14 for complex128 programs; 4e-7 for complex64 ones, whose entries are
// float32 roundings of cos and sin: the rotation by atan2(s, c) differs from
// the rounded matrix by less than float32's own rounding).
bool rotation_form(const C* m, double tol, int* mode, double* t, double* s, bool* neg) {
  const C a = m[0], b = m[1], cc = m[2], d = m[3];
  const bool real = a.im == 0 && b.im == 0 && cc.im == 0 && d.im == 0;
  double c, sn;
  if (real && a.re == d.re && b.re == -cc.re) {
    *mode = 0, c = a.re, sn = cc.re;
  } else if (real && a.re == -d.re && b.re == cc.re) {
    *mode = 1, c = a.re, sn = cc.re;
  } else if (a.re == d.re && a.im == 0 && d.im == 0 && b.re == 0 && cc.re == 0 && b.im == cc.im) {
    *mode = 2, c = a.re, sn = -b.im;
  } else {
    return false;
  }
  if (std::fabs(c * c + sn * sn - 1.0) > tol) return false;
  *neg = c < 0;
  if (*neg) c = -c, sn = -sn;
  *t = sn / (1.0 + c);
  *s = sn;
  return true;
}

// Reads and checks the planned gates of a pass (`who` names the entry point in
// errors): every qubit in range and given once, non-diagonal targets on tile
// bits, the entries each kind needs. No-ops are left out.
int parse_ops(int nqubits, const int* tile_bits, int nops, const int* op_desc, const double* op_data,
              const int64_t* data_offsets, std::vector<Op>& items, const char* who) {
  const std::string w = std::string(who) + ": ";
  uint64_t tmask = 0;
  for (int i = 0; i < kTileBits; ++i) {
    QSIM_CHECK_ARG(tile_bits[i] >= 0 && tile_bits[i] < nqubits && (i == 0 || tile_bits[i] > tile_bits[i - 1]),
                   w + "tile bits must ascend inside the register");
    tmask |= uint64_t(1) << tile_bits[i];
  }
  items.reserve(size_t(nops));
  for (int i = 0; i < nops; ++i) {
    const int* d = op_desc + size_t(i) * kDescInts;
    Op o;
    std::memset(&o, 0, sizeof(o));
    o.kind = d[0];
    o.nt = d[1];
    o.nc = d[2];
    QSIM_CHECK_ARG(o.kind >= kNoop && o.kind <= kDense, w + "bad op kind");
    QSIM_CHECK_ARG(o.nt >= 0 && o.nt <= kMaxTargets && o.nc >= 0 && o.nc <= kMaxControls,
                   w + "bad qubit counts");
    if (o.kind == kNoop) continue;
    uint64_t seen = 0;
    for (int k = 0; k < o.nt + o.nc; ++k) {
      const int q = k < o.nt ? d[4 + k] : d[9 + (k - o.nt)];
      QSIM_CHECK_ARG(q >= 0 && q < nqubits, w + "qubit out of range");
      const uint64_t bit = uint64_t(1) << (nqubits - 1 - q);
      QSIM_CHECK_ARG(!(seen & bit), w + "qubit given twice");
      seen |= bit;
      if (k < o.nt)
        o.t[k] = q;
      else
        o.c[k - o.nt] = q;
    }
    int need = 0;
    if (o.kind == kDiag) {
      QSIM_CHECK_ARG(o.nt <= 5, w + "diagonal on more than 5 targets");
      need = 1 << o.nt;
    } else if (o.kind == kDense) {
      QSIM_CHECK_ARG(o.nt >= 1 && o.nt <= 3, w + "dense gates in a pass act on 1..3 targets");
      need = (1 << o.nt) * (1 << o.nt);
    } else {
      QSIM_CHECK_ARG(o.nt == 2, w + "SWAP acts on 2 targets");
    }
    const int64_t off = data_offsets[i];
    QSIM_CHECK_ARG(need == 0 || off >= 0, w + "missing gate data");
    o.data = need ? reinterpret_cast<const C*>(op_data) + off : nullptr;
    o.ndata = need;
    for (int k = 0; k < o.nt; ++k) {
      const uint64_t bit = uint64_t(1) << (nqubits - 1 - o.t[k]);
      o.all_mask |= bit;
      if (o.kind != kDiag) {
        QSIM_CHECK_ARG(tmask & bit, w + "a non-diagonal target outside the tile bits");
        o.nd_mask |= bit;
      }
    }
    for (int k = 0; k < o.nc; ++k) o.all_mask |= uint64_t(1) << (nqubits - 1 - o.c[k]);
    items.push_back(o);
  }
  return QSIM_OK;
}

}  // namespace
