// Expectation values of Pauli sums, Hamiltonian-vector products and
// <bra|M|ket> inner products for gfx950, all accumulated in FP64.
//
// A Pauli string is i^{ny} X^x Z^z with bit masks x, z over amplitude
// indices (Y = i X Z). Then
//   (P psi)_i = i^{ny} (-1)^{popcount((i ^ x) & z)} psi_{i ^ x}
// and <psi|P|psi> pairs amplitude i0 (bit h of x clear, h = top bit of x) with
// i1 = i0 ^ x: A = conj(psi_i0) psi_i1 contributes
//   Re( i^{ny} ( (-1)^{|i1 & z|} A + (-1)^{|i0 & z|} conj(A) ) ).
// Strings with equal x share one pass over the state; x = 0 strings reduce
// |psi_i|^2 with their signs in one pass. This replaces the per-term einsum
// of Backend.exp_value_observable_symbolic (abstract.py:2946-3054).
//
// Reductions use a fixed grid and fixed-order trees, so results do not
// depend on scheduling (a request gives the same value alone or in a mix).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>

#include "qsim_common.h"

namespace qsim {

constexpr int kET = 256;
constexpr int kEBlocks = 1024;  // fixed grid of every reduction pass
constexpr int kMaxGroupTerms = 32;
constexpr int kESpread = 256;   // workgroups the items of a few tiles are spread over (one per CU)

struct PauliGroupArgs {
  uint64_t nwork;
  uint64_t x;      // flip mask of the group
  uint64_t hbit;   // top bit of x
  int hpos;
  int nterms;
  uint64_t z[kMaxGroupTerms];
  double c[kMaxGroupTerms];
  int ny[kMaxGroupTerms];
};

__device__ double block_sum(double v, double* lds) {
  lds[threadIdx.x] = v;
  __syncthreads();
  for (int off = kET / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) lds[threadIdx.x] += lds[threadIdx.x + off];
    __syncthreads();
  }
  return lds[0];
}

template <typename R>
__global__ __launch_bounds__(kET) void k_pauli_group(const cplx<R>* __restrict__ psi, const PauliGroupArgs a,
                                                     double* __restrict__ partial) {
  __shared__ double lds[kET];
  double acc = 0.0;
  const uint64_t stride = uint64_t(gridDim.x) * kET;
  for (uint64_t j = uint64_t(blockIdx.x) * kET + threadIdx.x; j < a.nwork; j += stride) {
    const uint64_t low = j & (a.hbit - 1);
    const uint64_t i0 = low | ((j ^ low) << 1);
    const uint64_t i1 = i0 ^ a.x;
    const cplx<R> u = psi[i0], v = psi[i1];
    // A = conj(u) * v
    const double are = double(u.re) * double(v.re) + double(u.im) * double(v.im);
    const double aim = double(u.re) * double(v.im) - double(u.im) * double(v.re);
    for (int t = 0; t < a.nterms; ++t) {
      const double s1 = (__popcll(i1 & a.z[t]) & 1) ? -1.0 : 1.0;
      const double s0 = (__popcll(i0 & a.z[t]) & 1) ? -1.0 : 1.0;
      // w = s1 A + s0 conj(A)
      const double wre = (s1 + s0) * are;
      const double wim = (s1 - s0) * aim;
      // Re(i^ny w)
      double re;
      switch (a.ny[t] & 3) {
        case 0: re = wre; break;
        case 1: re = -wim; break;
        case 2: re = -wre; break;
        default: re = wim; break;
      }
      acc += a.c[t] * re;
    }
  }
  const double tot = block_sum(acc, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// ---------------------------------------------------------------------------
// Many X masks per read of the state.
//
// One pass per X mask reads the whole state each time (the transverse-field
// Ising chain on 27 qubits: 28 passes of 0.39 ms). Here a workgroup holds a
// tile of 4096 amplitudes -- 16 per lane in registers, all of them in LDS --
// and forms every group whose mask flips tile bits only: the partner of
// amplitude i is i ^ x of the same tile, from the lane's own registers or
// from LDS. With the lowest 3 index bits in every tile (whole 128-byte lines)
// a pass covers 9 more flip bits, so that chain takes 3 passes: 10.9 -> 1.6 ms,
// 0.53 ms per 2 GiB read. A pass reads 16 bytes of LDS per amplitude and mask
// that is not one register bit, and two workgroups (64 KB of LDS each) share
// a CU, so loads and sums overlap only in part (complex64 takes the same time).
//
//   (P psi)_i = w(i) psi_{i ^ x},  w(i) = c i^ny (-1)^{|(i ^ x) & z|}
//
// The sign of a term factors into a tile part, a lane part and one of 16
// patterns over the registers: one bit per term and lane (the tile's bits come
// from one ballot), so no term's masks are read inside the loop over tiles.
// ---------------------------------------------------------------------------
constexpr int kPTileBits = 12;
constexpr int kPReg = 16;
constexpr int kPLaneBits = 8;     // local bits 0-7: the lane; 8-11: the register
constexpr int kPLowBits = 3;      // index bits in every tile
constexpr int kPMaxItems = 64;      // 48 beside more than 32 x = 0 terms (see PauliZ)
constexpr int kPMaxDiag = 64;

enum : uint32_t { kPImag = 1u << 16, kPFar = 1u << 17 };

// One or two terms of one X mask, their coefficients both real or both
// imaginary. A term's sign at amplitude i is a tile part times a lane part
// (one bit per term, see SignBits) times `pat`: bit r set where it is negative
// on register r.
struct PauliItem {
  uint32_t xl;      // flip mask on the local bits | flags
  uint16_t pat[2];
  double k[2];      // c (-1)^{|x & z|}, negated for ny = 2, 3
  uint64_t x;       // the whole mask, read where it leaves the tile
};

struct PauliTileArgs {
  uint64_t ntiles;
  uint64_t stride;  // amplitudes between the states of a batch (grid y)
  uint32_t valid;   // amplitudes of a tile that exist (registers below 12 qubits)
  int nitems, ndiag;
  int per;          // items per grid z (the terms of x = 0 belong to z = 0)
  int accumulate;   // APPLY: out += instead of out =
  uint8_t tbits[kPTileBits];  // index bit of local bit i, ascending
  uint8_t dcount[kPReg];      // x = 0 terms per register pattern, dk sorted by it
  PauliItem item[kPMaxItems];
  double dk[kPMaxDiag];
};

// z masks of the terms in bit order of the sign words: the items' terms from
// word 0 on (two bits per item), the first 32 x = 0 terms in word 4, the next 32
// in word 3, which the items past the 48th would take. So 64 terms of any kind
// fit one launch (kernel arguments end at 4 KB) and a complex64 product of 64
// terms is rounded once. The mask inside the lane bits sits in the top byte.
constexpr int kPWords = 5;
constexpr int kPZLaneShift = 56;
struct PauliZ {
  uint64_t z[32 * kPWords];
};
static_assert(QSIM_MAX_QUBITS <= kPZLaneShift && kPLaneBits <= 64 - kPZLaneShift, "masks of a term share a word");
static_assert(sizeof(PauliTileArgs) + sizeof(PauliZ) + 3 * sizeof(void*) <= 4096, "kernel arguments");

template <typename R>
__device__ __forceinline__ cplx<double> widen(cplx<R> v) {
  cplx<double> d;
  d.re = double(v.re);
  d.im = double(v.im);
  return d;
}

__device__ __forceinline__ double xor_sign(double k, uint32_t sign) {
  return __hiloint2double(int(uint32_t(__double2hiint(k)) ^ sign), __double2loint(k));
}

// Visits the lane's 16 (register, partner) pairs of one item.
template <bool FAR, typename R, typename F>
__device__ __forceinline__ void pauli_pairs(const cplx<R>* v, const cplx<R>* lds, const cplx<R>* psi, uint64_t first,
                                            const uint64_t* goff, const PauliItem& g, uint32_t lane, F&& f) {
  if constexpr (FAR) {
    if (g.xl & kPFar) {  // first: the index of the lane's register 0
      const uint64_t at = first ^ g.x;
#pragma unroll
      for (int r0 = 0; r0 < kPReg; r0 += 8) {
        cplx<R> u[8];  // eight loads in flight
#pragma unroll
        for (int r = 0; r < 8; ++r) u[r] = ld(psi, at ^ goff[r0 + r]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 8; ++r) f(r0 + r, widen(u[r]));
      }
      return;
    }
  }
  const uint32_t xl = g.xl & ((1u << kPTileBits) - 1);
  if (xl == (1u << kPLaneBits)) {
#pragma unroll
    for (int r = 0; r < kPReg; ++r) f(r, widen(v[r ^ 1]));
  } else if (xl == (2u << kPLaneBits)) {
#pragma unroll
    for (int r = 0; r < kPReg; ++r) f(r, widen(v[r ^ 2]));
  } else if (xl == (4u << kPLaneBits)) {
#pragma unroll
    for (int r = 0; r < kPReg; ++r) f(r, widen(v[r ^ 4]));
  } else if (xl == (8u << kPLaneBits)) {
#pragma unroll
    for (int r = 0; r < kPReg; ++r) f(r, widen(v[r ^ 8]));
  } else {
    const uint32_t at = lane ^ xl;  // (lane bits and register bits are disjoint)
#pragma unroll
    for (int r0 = 0; r0 < kPReg; r0 += 8) {
      cplx<R> u[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) u[r] = lds[at ^ (uint32_t(r0 + r) << kPLaneBits)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 8; ++r) f(r0 + r, widen(u[r]));
    }
  }
}

// Index bits contributed by local index u.
__device__ __forceinline__ uint64_t pauli_deposit(const PauliTileArgs& a, uint32_t u) {
  uint64_t i = 0;
#pragma unroll
  for (int b = 0; b < kPTileBits; ++b)
    if ((u >> b) & 1) i |= uint64_t(1) << a.tbits[b];
  return i;
}

// Energy (APPLY = false): partial[block] = sum over the block's tiles of
// Re conj(psi_i) w(i) psi_{i ^ x}. APPLY: out_i (+)= sum of w(i) psi_{i ^ x}
// and that sum beside it (masks that leave the tile read their partners from
// memory), one state of a batch per grid y; partial may be null.
template <typename R, bool APPLY>
__global__ __launch_bounds__(kET, 2) void k_pauli_tile(const cplx<R>* __restrict__ psi, cplx<R>* __restrict__ out,
                                                       const PauliTileArgs a, const PauliZ zz,
                                                       double* __restrict__ partial) {
  __shared__ cplx<R> lds[1 << kPTileBits];
  __shared__ double red[kET];
  const uint32_t lane = threadIdx.x;
  psi += uint64_t(blockIdx.y) * a.stride;
  const uint64_t lane_off = pauli_deposit(a, lane);
  uint64_t goff[kPReg];
#pragma unroll
  for (int r = 0; r < kPReg; ++r) goff[r] = pauli_deposit(a, uint32_t(r) << kPLaneBits);
  auto load = [&](uint64_t tile, cplx<R>* v) {
    const uint64_t at = insert_zeros(tile, a.tbits, kPTileBits) | lane_off;
    if (a.valid == (1u << kPTileBits)) {
#pragma unroll
      for (int r = 0; r < kPReg; ++r) v[r] = ld(psi, at | goff[r]);
    } else {  // a register below 12 qubits: the amplitudes past it are zero (amplitude 0 is read in their place)
#pragma unroll
      for (int r = 0; r < kPReg; ++r) {
        const bool there = (lane | (uint32_t(r) << kPLaneBits)) < a.valid;
        v[r] = ld(psi, there ? at | goff[r] : 0);
        v[r].re = there ? v[r].re : R(0);
        v[r].im = there ? v[r].im : R(0);
      }
    }
  };
  const int i0 = int(blockIdx.z) * a.per;
  const int i1 = i0 + a.per < a.nitems ? i0 + a.per : a.nitems;
  const bool diag = a.ndiag > 0 && blockIdx.z == 0;
  // one sign bit per term: the lane's part once, the tile's part per tile (a
  // wave's lane t forms term t's)
  uint32_t lane_sign[kPWords];
  uint64_t zo[(kPWords + 1) / 2];
#pragma unroll
  for (int w = 0; w < kPWords; ++w) {
    lane_sign[w] = 0;
    const int items = 2 * a.nitems - 32 * w, diags = a.ndiag - 32 * (4 - w);
    const int cnt = w == 4 ? a.ndiag : (w == 3 && diags > items ? diags : items);
    for (int t = 0; t < 32 && t < cnt; ++t)
      lane_sign[w] |= uint32_t(__popc(lane & uint32_t(zz.z[32 * w + t] >> kPZLaneShift)) & 1) << t;
  }
#pragma unroll
  for (int h = 0; h < (kPWords + 1) / 2; ++h) {
    const int t = 64 * h + int(lane & 63);
    zo[h] = t < 32 * kPWords ? zz.z[t] : 0;
  }
  double acc = 0.0;
  cplx<R> v[kPReg];
  for (uint64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    load(tile, v);
    const uint64_t origin = insert_zeros(tile, a.tbits, kPTileBits);
    uint32_t sign[kPWords];
#pragma unroll
    for (int h = 0; h < (kPWords + 1) / 2; ++h) {
      const uint64_t odd = __ballot(__popcll(origin & zo[h]) & 1);
      sign[2 * h] = lane_sign[2 * h] ^ uint32_t(odd);
      if (2 * h + 1 < kPWords) sign[2 * h + 1] = lane_sign[2 * h + 1] ^ uint32_t(odd >> 32);
    }
#pragma unroll
    for (int r = 0; r < kPReg; ++r) lds[lane | (uint32_t(r) << kPLaneBits)] = v[r];
    __syncthreads();
    cplx<double> o[APPLY ? kPReg : 1];
    if constexpr (APPLY) {
#pragma unroll
      for (int r = 0; r < kPReg; ++r) o[r] = cplx<double>{0.0, 0.0};
    }
    if (diag) {
      // coefficients per register pattern, then one 16-point Walsh-Hadamard
      // transform: w on the lane's 16 amplitudes
      double w[kPReg];
      int t = 0;
      uint32_t word = sign[4];
#pragma unroll
      for (int k = 0; k < kPReg; ++k) {
        w[k] = 0.0;
        for (int left = a.dcount[k]; left > 0; --left) {
          w[k] += xor_sign(a.dk[t], word << 31);
          word = ++t == 32 ? sign[3] : word >> 1;
        }
      }
#pragma unroll
      for (int h = 1; h < kPReg; h <<= 1)
#pragma unroll
        for (int r = 0; r < kPReg; ++r)
          if (!(r & h)) {
            const double x = w[r], y = w[r | h];
            w[r] = x + y;
            w[r | h] = x - y;
          }
#pragma unroll
      for (int r = 0; r < kPReg; ++r) {
        const cplx<double> u = widen(v[r]);
        if constexpr (APPLY) {
          o[r].re = w[r] * u.re;
          o[r].im = w[r] * u.im;
        } else {
          acc = __builtin_fma(w[r], __builtin_fma(u.re, u.re, u.im * u.im), acc);
        }
      }
    }
    PauliItem next = a.item[i0 < i1 ? i0 : 0];
    uint32_t word = sign[0];
    if (i0 >= 48)
      word = sign[3];
    else if (i0 >= 32)
      word = sign[2];
    else if (i0 >= 16)
      word = sign[1];
    word >>= 2 * (i0 & 15);
    for (int i = i0; i < i1; ++i) {
      const PauliItem g = next;  // read one item ahead
      next = a.item[i + 1 < i1 ? i + 1 : i];
      const uint32_t s0 = word << 31, s1 = (word << 30) & 0x80000000u;
      word >>= 2;
      if (((i + 1) & 15) == 0) word = i == 15 ? sign[1] : (i == 31 ? sign[2] : sign[3]);
      // (products of the lane's own amplitudes are formed where they are used,
      // not kept in registers from one item to the next)
#pragma unroll
      for (int r = 0; r < kPReg; ++r) asm volatile("" : "+v"(v[r].re), "+v"(v[r].im));
      double k0 = xor_sign(g.k[0], s0);
      const double k1 = xor_sign(g.k[1], s1);
      const bool same = (g.pat[0] | g.pat[1]) == 0;
      if (same) k0 += k1;  // (k[1] = 0 of a single term)
      const uint32_t p0 = g.pat[0], p1 = g.pat[1];
      auto weight = [&](int r) {
        return xor_sign(k0, p0 << (31 - r) & 0x80000000u) + xor_sign(k1, p1 << (31 - r) & 0x80000000u);
      };
      if constexpr (!APPLY) {
        // Re(w B) with B = conj(psi_i) psi_{i ^ x}: w Re B, or -w Im B for imaginary w
        double s[4] = {0.0, 0.0, 0.0, 0.0};  // four chains of additions
        if (g.xl & kPImag) {
          pauli_pairs<false>(v, lds, psi, origin | lane_off, goff, g, lane, [&](int r, cplx<double> u) {
            const double b = __builtin_fma(double(v[r].im), u.re, -(double(v[r].re) * u.im));
            s[r & 3] = __builtin_fma(same ? k0 : weight(r), b, s[r & 3]);
          });
          acc += (s[0] + s[1]) + (s[2] + s[3]);
        } else if (same) {
          pauli_pairs<false>(v, lds, psi, origin | lane_off, goff, g, lane, [&](int r, cplx<double> u) {
            s[r & 3] = __builtin_fma(double(v[r].re), u.re, __builtin_fma(double(v[r].im), u.im, s[r & 3]));
          });
          acc = __builtin_fma(k0, (s[0] + s[1]) + (s[2] + s[3]), acc);
        } else {
          pauli_pairs<false>(v, lds, psi, origin | lane_off, goff, g, lane, [&](int r, cplx<double> u) {
            const double b = __builtin_fma(double(v[r].re), u.re, double(v[r].im) * u.im);
            s[r & 3] = __builtin_fma(weight(r), b, s[r & 3]);
          });
          acc += (s[0] + s[1]) + (s[2] + s[3]);
        }
      } else {
        if (g.xl & kPImag) {
          pauli_pairs<true>(v, lds, psi, origin | lane_off, goff, g, lane, [&](int r, cplx<double> u) {
            const double k = same ? k0 : weight(r);
            o[r].re = __builtin_fma(-k, u.im, o[r].re);
            o[r].im = __builtin_fma(k, u.re, o[r].im);
          });
        } else if (same) {
          pauli_pairs<true>(v, lds, psi, origin | lane_off, goff, g, lane, [&](int r, cplx<double> u) {
            o[r].re = __builtin_fma(k0, u.re, o[r].re);
            o[r].im = __builtin_fma(k0, u.im, o[r].im);
          });
        } else {
          pauli_pairs<true>(v, lds, psi, origin | lane_off, goff, g, lane, [&](int r, cplx<double> u) {
            const double k = weight(r);
            o[r].re = __builtin_fma(k, u.re, o[r].re);
            o[r].im = __builtin_fma(k, u.im, o[r].im);
          });
        }
      }
    }
    if constexpr (APPLY) {
      cplx<R>* dst = out + uint64_t(blockIdx.y) * a.stride + (origin | lane_off);
#pragma unroll
      for (int r = 0; r < kPReg; ++r) {
        if ((lane | (uint32_t(r) << kPLaneBits)) >= a.valid) continue;
        acc = __builtin_fma(double(v[r].re), o[r].re, __builtin_fma(double(v[r].im), o[r].im, acc));
        if (a.accumulate) {
          o[r].re += double(dst[goff[r]].re);
          o[r].im += double(dst[goff[r]].im);
        }
        dst[goff[r]].re = R(o[r].re);
        dst[goff[r]].im = R(o[r].im);
      }
    }
    __syncthreads();
  }
  const double tot = block_sum(acc, red);
  if (threadIdx.x == 0 && partial != nullptr)
    partial[(uint64_t(blockIdx.z) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = tot;
}

// A launch being filled: its arguments, and the z masks of its terms.
struct PauliBatch {
  PauliTileArgs a;
  PauliZ zz;
  uint64_t item_z[kPMaxItems][2];
  uint64_t diag_z[kPMaxDiag];
  double diag_k[kPMaxDiag];

  void clear() { std::memset(this, 0, sizeof(*this)); }
  bool empty() const { return a.nitems == 0 && a.ndiag == 0; }

  // Whether a group (at most 32 terms of one X mask) still fits.
  bool fits(const PauliGroupArgs& p) const {
    int odd = 0;
    for (int i = 0; i < p.nterms; ++i) odd += p.ny[i] & 1;
    const int even = p.nterms - odd;
    const int diags = a.ndiag + (p.x == 0 ? even : 0);
    const int items = a.nitems + (odd + 1) / 2 + (p.x == 0 ? 0 : (even + 1) / 2);
    return diags <= kPMaxDiag && items <= (diags > 32 ? kPMaxItems - 16 : kPMaxItems);
  }

  void append(const PauliGroupArgs& p) {
    for (int odd = 0; odd < 2; ++odd) {
      int used = 2;  // terms in the current item
      for (int i = 0; i < p.nterms; ++i) {
        // (a diagonal product with odd ny is anti-Hermitian: its expectation's
        // real part is zero, its product with the state an imaginary weight)
        if ((p.ny[i] & 1) != odd) continue;
        const bool neg = ((p.ny[i] & 2) != 0) != ((__builtin_popcountll(p.x & p.z[i]) & 1) != 0);
        const double k = neg ? -p.c[i] : p.c[i];
        if (p.x == 0 && !odd) {
          diag_z[a.ndiag] = p.z[i];
          diag_k[a.ndiag++] = k;
          continue;
        }
        if (used == 2) {
          PauliItem& g = a.item[a.nitems++];
          g.x = p.x;
          g.xl = odd ? kPImag : 0;
          used = 0;
        }
        item_z[a.nitems - 1][used] = p.z[i];
        a.item[a.nitems - 1].k[used++] = k;
      }
    }
  }

  // Fixes the tile bits (`tmask` and the lowest free index bits up to 12) and
  // writes the local forms of the terms.
  void finish(int n, uint64_t tmask) {
    const int nb = n < kPTileBits ? n : kPTileBits;
    int have = __builtin_popcountll(tmask);
    for (int b = 0; b < n && have < nb; ++b)
      if (!((tmask >> b) & 1)) tmask |= uint64_t(1) << b, ++have;
    int k = 0;
    for (int b = 0; b < 64; ++b)
      if ((tmask >> b) & 1) a.tbits[k++] = uint8_t(b);
    for (; k < kPTileBits; ++k) a.tbits[k] = uint8_t(k);  // below 12 qubits: bits past the register, never loaded
    a.valid = uint32_t(1) << nb;
    a.ntiles = uint64_t(1) << (n - nb);
    auto localize = [&](uint64_t m) {
      uint32_t l = 0;
      for (int i = 0; i < nb; ++i)
        if ((m >> a.tbits[i]) & 1) l |= uint32_t(1) << i;
      return l;
    };
    auto pattern = [&](uint64_t z) {
      uint32_t p = 0;
      for (int r = 0; r < kPReg; ++r)
        if (__builtin_popcount(uint32_t(r) & (localize(z) >> kPLaneBits)) & 1) p |= 1u << r;
      return uint16_t(p);
    };
    auto put = [&](int bit, uint64_t z) {
      zz.z[bit] = (z & ~tmask) | uint64_t(localize(z) & ((1u << kPLaneBits) - 1)) << kPZLaneShift;
    };
    int d = 0;
    for (int c = 0; c < kPReg; ++c) {
      const int first = d;
      for (int i = 0; i < a.ndiag; ++i)
        if ((localize(diag_z[i]) >> kPLaneBits) == uint32_t(c)) {
          a.dk[d] = diag_k[i];
          put(d < 32 ? 128 + d : 64 + d, diag_z[i]);
          ++d;
        }
      a.dcount[c] = uint8_t(d - first);
    }
    for (int i = 0; i < a.nitems; ++i) {
      PauliItem& g = a.item[i];
      if (g.x & ~tmask)
        g.xl |= kPFar;
      else
        g.xl |= localize(g.x);
      for (int t = 0; t < 2; ++t) {
        g.pat[t] = pattern(item_z[i][t]);
        put(2 * i + t, item_z[i][t]);
      }
    }
  }
};

// out[b] = the sum of state b's partials: `count` of each of `nrow` launches,
// row r of state b at partial[(r * gridDim.x + b) * count].
__global__ __launch_bounds__(kET) void k_sum_partials(const double* __restrict__ partial, int64_t count, int nrow,
                                                      double* __restrict__ out) {
  __shared__ double lds[kET];
  double acc = 0.0;
  for (int r = 0; r < nrow; ++r)
    for (int64_t i = threadIdx.x; i < count; i += kET)
      acc += partial[(int64_t(r) * gridDim.x + blockIdx.x) * count + i];
  const double tot = block_sum(acc, lds);
  if (threadIdx.x == 0) out[blockIdx.x] = tot;
}

static int grid_for(uint64_t nwork) {
  const uint64_t b = (nwork + kET - 1) / kET;
  return int(b < kEBlocks ? (b < 1 ? 1 : b) : kEBlocks);
}

// The launches of a term table, in the order every entry point uses: the
// distinct x masks in ascending order, each split into chunks of at most
// kMaxGroupTerms terms in table order. Found by repeated minimum scans, so no
// container is allocated (the no-allocation entry point shares it).
template <typename F>
static void for_each_group(int nterms, const uint64_t* xm, const uint64_t* zm, const int* ny, const double* c,
                           F&& visit) {
  bool have = false;
  uint64_t cur = 0;
  for (int t = 0; t < nterms; ++t)
    if (!have || xm[t] < cur) cur = xm[t], have = true;
  while (have) {
    PauliGroupArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = cur;
    for (int t = 0; t < nterms; ++t) {
      if (xm[t] != cur) continue;
      a.z[a.nterms] = zm[t];
      a.c[a.nterms] = c[t];
      a.ny[a.nterms] = ny[t];
      if (++a.nterms == kMaxGroupTerms) {
        visit(a);
        a.nterms = 0;
      }
    }
    if (a.nterms > 0) visit(a);
    bool next = false;
    uint64_t nxt = 0;
    for (int t = 0; t < nterms; ++t)
      if (xm[t] > cur && (!next || xm[t] < nxt)) nxt = xm[t], next = true;
    have = next;
    cur = nxt;
  }
}

// Launches the group passes into partial[0 ..) and the final fixed-order sum;
// the partial buffer must hold ngroups * kEBlocks doubles (checked first).
template <typename R>
static int expval_impl(const void* state, int n, int nterms, const uint64_t* xm, const uint64_t* zm,
                       const int* ny, const double* c, double* out, void* ws, size_t ws_bytes, hipStream_t s,
                       const char* who) {
  size_t ngroups = 0;
  for_each_group(nterms, xm, zm, ny, c, [&](const PauliGroupArgs&) { ++ngroups; });
  if (ngroups * kEBlocks * sizeof(double) > ws_bytes) {
    set_error(std::string(who) + ": workspace too small for " + std::to_string(ngroups) +
              " term groups (distinct X masks, 32 terms per group)");
    return QSIM_EINVAL;
  }
  double* partial = reinterpret_cast<double*>(ws);
  int64_t used = 0;
  int rc = QSIM_OK;
  const uint64_t low = (uint64_t(1) << std::min(n, kPLowBits)) - 1;
  const int nb = std::min(n, kPTileBits);
  PauliBatch cur;
  cur.clear();
  uint64_t tmask = low;
  auto launched = [&](int blocks) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      set_error(std::string(who) + ": launch failed: " + hipGetErrorString(e));
      rc = QSIM_EHIP;
      return;
    }
    used += blocks;
  };
  auto flush = [&]() {
    if (cur.empty()) return;
    cur.finish(n, tmask);
    // few tiles: the items are spread over more workgroups
    const int blocks = int(std::min<uint64_t>(cur.a.ntiles, kEBlocks));
    int parts = std::max(1, std::min(cur.a.nitems, kESpread / blocks));
    cur.a.per = std::max(1, (cur.a.nitems + parts - 1) / parts);
    parts = std::max(1, (cur.a.nitems + cur.a.per - 1) / cur.a.per);
    hipLaunchKernelGGL((k_pauli_tile<R, false>), dim3(unsigned(blocks), 1, unsigned(parts)), dim3(kET), 0, s,
                       reinterpret_cast<const cplx<R>*>(state), static_cast<cplx<R>*>(nullptr), cur.a, cur.zz,
                       partial + used);
    launched(blocks * parts);
    cur.clear();
    tmask = low;
  };
  // groups in ascending mask order share a tile pass while their flip bits
  // (and the lowest bits) fit in 12; a mask that flips too many bits for any
  // tile takes a pass of its own
  for_each_group(nterms, xm, zm, ny, c, [&](const PauliGroupArgs& g) {
    if (rc != QSIM_OK) return;
    if (__builtin_popcountll(g.x | low) > nb) {
      PauliGroupArgs a = g;
      a.hpos = 63 - __builtin_clzll(a.x);
      a.hbit = uint64_t(1) << a.hpos;
      a.nwork = uint64_t(1) << (n - 1);
      const int blocks = grid_for(a.nwork);
      hipLaunchKernelGGL(k_pauli_group<R>, dim3(blocks), dim3(kET), 0, s, reinterpret_cast<const cplx<R>*>(state), a,
                         partial + used);
      launched(blocks);
      return;
    }
    if (__builtin_popcountll(tmask | g.x) > nb || !cur.fits(g)) flush();
    if (rc != QSIM_OK) return;
    tmask |= g.x;
    cur.append(g);
  });
  if (rc == QSIM_OK) flush();
  if (rc != QSIM_OK) return rc;
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kET), 0, s, partial, used, 1, out);
  QSIM_CHECK_LAUNCH();
  return QSIM_OK;
}

// ---------------------------------------------------------------------------
// out = sum_t c_t P_t psi of one state of few tiles or by few terms (gather
// form, one output amplitude per thread: more workgroups than tiles; 16 qubits:
// 15 us against 24 us by tiles; see tiles_pay)
// ---------------------------------------------------------------------------
struct PauliApplyArgs {
  uint64_t n;
  int nterms;
  uint64_t x[64];
  uint64_t z[64];
  double c[64];
  int ny[64];
};

template <typename R>
__global__ __launch_bounds__(kET) void k_pauli_apply(const cplx<R>* __restrict__ psi, cplx<R>* __restrict__ out,
                                                     const PauliApplyArgs a, int accumulate) {
  const uint64_t i = block_id() * kET + threadIdx.x;
  if (i >= a.n) return;
  double re = 0.0, im = 0.0;
  if (accumulate) {
    re = double(out[i].re);
    im = double(out[i].im);
  }
  for (int t = 0; t < a.nterms; ++t) {
    const uint64_t j = i ^ a.x[t];
    const cplx<R> v = psi[j];
    const double sgn = (__popcll(j & a.z[t]) & 1) ? -a.c[t] : a.c[t];
    double vr = sgn * double(v.re), vi = sgn * double(v.im);
    switch (a.ny[t] & 3) {  // multiply by i^ny
      case 0: break;
      case 1: { const double tr = -vi; vi = vr; vr = tr; } break;
      case 2: vr = -vr; vi = -vi; break;
      default: { const double tr = vi; vi = -vr; vr = tr; } break;
    }
    re += vr;
    im += vi;
  }
  out[i].re = R(re);
  out[i].im = R(im);
}

// ---------------------------------------------------------------------------
// out = sum_t c_t P_t psi for a batch of states, and <psi|out> beside it
// ---------------------------------------------------------------------------
// Launches of a term table: at most this many (a launch that is full holds 64
// terms or more, see PauliBatch::fits).
static int apply_launches(int nterms) { return 1 + nterms / 64; }

// Whether one state of 20 qubits or more (as many tiles as CUs) is cheaper by
// tiles than by k_pauli_apply. That one reads a partner per term and amplitude;
// a tile pass costs more before its first term and a little more for each mask
// that leaves the tile, but next to nothing for a term on the lowest 12 index
// bits and for further terms of one mask. Equal at so many
//   qubits                         20      22      24     27
//   terms in the tile, complex128  18-30   10-13   6-9    4-6   (diagonal ones to X)
//                      complex64   8-20    5-10    2-5    1
//   masks outside it, complex64    > 32    24      16     8     (complex128: none)
// (24 qubits, complex128: one X 89 us against 133 us by tiles, 24 Z pairs 319 us
// against 138 us).
static bool tiles_pay(int n, int dtype, int nterms, const uint64_t* xm, const uint64_t* zm, const int* ny,
                      const double* c) {
  int near = 0, again = 0, masks = 0;  // terms in the tile; further terms of masks outside it, and those masks
  uint64_t last = 0;
  for_each_group(nterms, xm, zm, ny, c, [&](const PauliGroupArgs& g) {
    if (!(g.x >> kPTileBits)) {
      near += g.nterms;
      return;
    }
    masks += g.x != last;
    again += g.nterms - (g.x != last);
    last = g.x;
  });
  // (a state below 24 qubits, complex64 22, stays in cache between its terms)
  const int small = std::max(0, 27 - n);
  if (dtype == QSIM_C128) return near + (n < 24 ? 1 : 5) * again - masks >= 4 + 2 * small;
  return 2 * near + (n < 22 ? 2 : 6) * again + masks - (masks > 0 ? 8 : 0) >= 2 + 3 * small;
}

template <typename R>
static int apply_impl(const void* state, int nbatch, int n, int nterms, const uint64_t* xm, const uint64_t* zm,
                      const int* ny, const double* c, void* out, double* energies, double* partial, hipStream_t s,
                      const char* who) {
  PauliBatch cur;
  cur.clear();
  int rc = QSIM_OK, launches = 0, blocks = 0;
  auto flush = [&]() {
    if (cur.empty()) return;
    cur.finish(n, 0);
    cur.a.stride = uint64_t(1) << n;
    cur.a.accumulate = launches > 0;
    cur.a.per = std::max(1, cur.a.nitems);
    blocks = int(std::min<uint64_t>(cur.a.ntiles, kEBlocks));
    double* to = energies ? partial + size_t(launches) * size_t(nbatch) * size_t(blocks) : nullptr;
    hipLaunchKernelGGL((k_pauli_tile<R, true>), dim3(unsigned(blocks), unsigned(nbatch)), dim3(kET), 0, s,
                       reinterpret_cast<const cplx<R>*>(state), reinterpret_cast<cplx<R>*>(out), cur.a, cur.zz, to);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      set_error(std::string(who) + ": launch failed: " + hipGetErrorString(e));
      rc = QSIM_EHIP;
    }
    ++launches;
    cur.clear();
  };
  for_each_group(nterms, xm, zm, ny, c, [&](const PauliGroupArgs& g) {
    // a group is split where a launch is full: each launch rounds the product
    // to the state's type, so no launch leaves with fewer terms than it can hold
    for (int from = 0; from < g.nterms && rc == QSIM_OK;) {
      PauliGroupArgs part = g;
      for (part.nterms = g.nterms - from; part.nterms > 0; --part.nterms) {
        std::copy(g.z + from, g.z + from + part.nterms, part.z);
        std::copy(g.c + from, g.c + from + part.nterms, part.c);
        std::copy(g.ny + from, g.ny + from + part.nterms, part.ny);
        if (cur.fits(part)) break;
      }
      if (part.nterms == 0)
        flush();
      else
        cur.append(part);
      from += part.nterms;
    }
  });
  if (rc == QSIM_OK) flush();
  if (rc != QSIM_OK || !energies) return rc;
  hipLaunchKernelGGL(k_sum_partials, dim3(unsigned(nbatch)), dim3(kET), 0, s, partial, int64_t(blocks), launches,
                     energies);
  QSIM_CHECK_LAUNCH();
  return QSIM_OK;
}

// ---------------------------------------------------------------------------
// Re <bra| M |ket> on targets under controls
// ---------------------------------------------------------------------------
template <typename R, int NT>
struct InnerArgs {
  uint64_t nwork;
  uint64_t cmask;
  uint64_t off[1 << NT];
  cplx<R> m[(1 << NT) * (1 << NT)];
  int nfixed;
  uint8_t pos[kMaxFixed];
};

template <typename R, int NT>
__global__ __launch_bounds__(kET) void k_inner(const cplx<R>* __restrict__ bra, const cplx<R>* __restrict__ ket,
                                               const InnerArgs<R, NT> a, double* __restrict__ partial) {
  __shared__ double lds[kET];
  constexpr int D = 1 << NT;
  double acc = 0.0;
  const uint64_t stride = uint64_t(gridDim.x) * kET;
  for (uint64_t j = uint64_t(blockIdx.x) * kET + threadIdx.x; j < a.nwork; j += stride) {
    const uint64_t base = insert_zeros(j, a.pos, a.nfixed) | a.cmask;
    cplx<R> k[D];
#pragma unroll
    for (int c = 0; c < D; ++c) k[c] = ket[base | a.off[c]];
#pragma unroll
    for (int r = 0; r < D; ++r) {
      double yr = 0.0, yi = 0.0;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        yr += double(a.m[r * D + c].re) * double(k[c].re) - double(a.m[r * D + c].im) * double(k[c].im);
        yi += double(a.m[r * D + c].re) * double(k[c].im) + double(a.m[r * D + c].im) * double(k[c].re);
      }
      const cplx<R> b = bra[base | a.off[r]];
      acc += double(b.re) * yr + double(b.im) * yi;  // Re(conj(b) y)
    }
  }
  const double tot = block_sum(acc, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

template <typename R, int NT>
static int launch_inner(const void* bra, const void* ket, int n, const int* targets, const int* controls, int nc,
                        const void* matrix, double* out, double* partial, hipStream_t s) {
  InnerArgs<R, NT> a;
  std::memset(&a, 0, sizeof(a));
  a.nfixed = sorted_positions(n, controls, nc, targets, NT, a.pos);
  a.nwork = uint64_t(1) << (n - a.nfixed);
  for (int i = 0; i < nc; ++i) a.cmask |= uint64_t(1) << (n - 1 - controls[i]);
  for (int r = 0; r < (1 << NT); ++r) {
    uint64_t off = 0;
    for (int t = 0; t < NT; ++t)
      if ((r >> (NT - 1 - t)) & 1) off |= uint64_t(1) << (n - 1 - targets[t]);
    a.off[r] = off;
  }
  std::memcpy(a.m, matrix, sizeof(a.m));
  const int blocks = grid_for(a.nwork);
  hipLaunchKernelGGL((k_inner<R, NT>), dim3(blocks), dim3(kET), 0, s, reinterpret_cast<const cplx<R>*>(bra),
                     reinterpret_cast<const cplx<R>*>(ket), a, partial);
  QSIM_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kET), 0, s, partial, int64_t(blocks), 1, out);
  QSIM_CHECK_LAUNCH();
  return QSIM_OK;
}

// ---------------------------------------------------------------------------
// Scratch for callers that cannot allocate (qsim_expval_pauli_noalloc): the
// per-block partial sums of up to kNoAllocGroups term groups in a file-scope
// device array. Each GPU holds its own copy (512 KiB) until the process ends;
// its address on a device comes from hipGetSymbolAddress, taken once per
// device with that device current. The array's name in host code is only a
// handle for that call, never a device address.
// ---------------------------------------------------------------------------
constexpr int kNoAllocGroups = 64;
constexpr int kNoAllocDevices = 64;
__device__ __align__(256) double scratch[kNoAllocGroups * kEBlocks];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kNoAllocDevices];  // per device, set once under g_scratch_mu

static int scratch_on_current_device(void* stream, double** out, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error(std::string(who) + ": hipGetDevice: " + hipGetErrorString(e));
    return QSIM_EHIP;
  }
  if (dev < 0 || dev >= kNoAllocDevices) {
    set_error(std::string(who) + ": device ordinal out of range");
    return QSIM_EINVAL;
  }
  if (stream != nullptr) {
    hipDevice_t sdev = -1;
    e = hipStreamGetDevice(reinterpret_cast<hipStream_t>(stream), &sdev);
    if (e != hipSuccess) {
      set_error(std::string(who) + ": hipStreamGetDevice: " + hipGetErrorString(e));
      return QSIM_EHIP;
    }
    if (int(sdev) != dev) {
      set_error(std::string(who) + ": the stream belongs to another device than the current one");
      return QSIM_EINVAL;
    }
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error(std::string(who) + ": hipGetSymbolAddress(scratch): " + hipGetErrorString(e));
      return QSIM_EHIP;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = reinterpret_cast<double*>(g_scratch_ptr[dev]);
  return QSIM_OK;
}

}  // namespace qsim

using namespace qsim;

extern "C" {

size_t qsim_expval_workspace(int nqubits, int nterms) {
  (void)nqubits;
  if (nterms < 1) nterms = 1;
  return size_t(nterms) * kEBlocks * sizeof(double);
}

int qsim_expval_pauli(const void* state, int nqubits, int dtype, int nterms, const uint64_t* xmasks,
                      const uint64_t* zmasks, const int* ny, const double* coeffs, double* out, void* workspace,
                      size_t workspace_bytes, void* stream) {
  clear_error();
  QSIM_CHECK_ARG(state != nullptr && out != nullptr && workspace != nullptr, "qsim_expval_pauli: null pointer");
  QSIM_CHECK_ARG(dtype == QSIM_C128 || dtype == QSIM_C64, "qsim_expval_pauli: bad dtype");
  QSIM_CHECK_ARG(nqubits >= 1 && nqubits <= QSIM_MAX_QUBITS, "qsim_expval_pauli: nqubits out of range");
  QSIM_CHECK_ARG(nterms >= 1 && xmasks && zmasks && ny && coeffs, "qsim_expval_pauli: bad term table");
  const uint64_t full = (nqubits == 64) ? ~uint64_t(0) : ((uint64_t(1) << nqubits) - 1);
  for (int t = 0; t < nterms; ++t)
    QSIM_CHECK_ARG((xmasks[t] & ~full) == 0 && (zmasks[t] & ~full) == 0, "qsim_expval_pauli: mask out of range");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == QSIM_C128)
    return expval_impl<double>(state, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, workspace, workspace_bytes, s,
                               "qsim_expval_pauli");
  return expval_impl<float>(state, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, workspace, workspace_bytes, s,
                            "qsim_expval_pauli");
}

int qsim_expval_pauli_noalloc(const void* state, int nqubits, int dtype, int nterms, const uint64_t* xmasks,
                              const uint64_t* zmasks, const int* ny, const double* coeffs, double* out,
                              void* stream) {
  clear_error();
  const char* who = "qsim_expval_pauli_noalloc";
  QSIM_CHECK_ARG(state != nullptr && out != nullptr, "qsim_expval_pauli_noalloc: null pointer");
  QSIM_CHECK_ARG(dtype == QSIM_C128 || dtype == QSIM_C64, "qsim_expval_pauli_noalloc: bad dtype");
  QSIM_CHECK_ARG(nqubits >= 1 && nqubits <= QSIM_MAX_QUBITS, "qsim_expval_pauli_noalloc: nqubits out of range");
  QSIM_CHECK_ARG(nterms >= 1 && xmasks && zmasks && ny && coeffs, "qsim_expval_pauli_noalloc: bad term table");
  const uint64_t full = (uint64_t(1) << nqubits) - 1;
  for (int t = 0; t < nterms; ++t)
    QSIM_CHECK_ARG((xmasks[t] & ~full) == 0 && (zmasks[t] & ~full) == 0,
                   "qsim_expval_pauli_noalloc: mask out of range");
  size_t ngroups = 0;
  for_each_group(nterms, xmasks, zmasks, ny, coeffs, [&](const PauliGroupArgs&) { ++ngroups; });
  if (ngroups > size_t(kNoAllocGroups)) {
    set_error("qsim_expval_pauli_noalloc: " + std::to_string(ngroups) + " term groups (distinct X masks, 32 terms " +
              "per group) exceed the maximum of " + std::to_string(kNoAllocGroups) +
              "; use qsim_expval_pauli with a workspace");
    return QSIM_EINVAL;
  }
  double* ptr = nullptr;
  const int rc = scratch_on_current_device(stream, &ptr, who);
  if (rc != QSIM_OK) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const size_t bytes = sizeof(double) * size_t(kNoAllocGroups) * size_t(kEBlocks);
  if (dtype == QSIM_C128)
    return expval_impl<double>(state, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, ptr, bytes, s, who);
  return expval_impl<float>(state, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, ptr, bytes, s, who);
}

int qsim_expval_noalloc_max_groups(void) { return kNoAllocGroups; }

int qsim_apply_pauli_sum(const void* state, int nqubits, int dtype, int nterms, const uint64_t* xmasks,
                         const uint64_t* zmasks, const int* ny, const double* coeffs, void* out, void* stream) {
  clear_error();
  QSIM_CHECK_ARG(state != nullptr && out != nullptr && state != out, "qsim_apply_pauli_sum: bad pointers");
  QSIM_CHECK_ARG(dtype == QSIM_C128 || dtype == QSIM_C64, "qsim_apply_pauli_sum: bad dtype");
  QSIM_CHECK_ARG(nqubits >= 1 && nqubits <= QSIM_MAX_QUBITS, "qsim_apply_pauli_sum: nqubits out of range");
  QSIM_CHECK_ARG(nterms >= 1 && xmasks && zmasks && ny && coeffs, "qsim_apply_pauli_sum: bad term table");
  const uint64_t full = (uint64_t(1) << nqubits) - 1;
  for (int t = 0; t < nterms; ++t)
    QSIM_CHECK_ARG((xmasks[t] & ~full) == 0 && (zmasks[t] & ~full) == 0, "qsim_apply_pauli_sum: mask out of range");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (nqubits < kPTileBits + 8 || !tiles_pay(nqubits, dtype, nterms, xmasks, zmasks, ny, coeffs)) {
    const uint64_t N = uint64_t(1) << nqubits;
    for (int t0 = 0; t0 < nterms; t0 += 64) {
      PauliApplyArgs a;
      std::memset(&a, 0, sizeof(a));
      a.n = N;
      a.nterms = std::min(64, nterms - t0);
      for (int t = 0; t < a.nterms; ++t) {
        a.x[t] = xmasks[t0 + t];
        a.z[t] = zmasks[t0 + t];
        a.c[t] = coeffs[t0 + t];
        a.ny[t] = ny[t0 + t];
      }
      const int acc = t0 > 0 ? 1 : 0;
      if (dtype == QSIM_C128)
        hipLaunchKernelGGL(k_pauli_apply<double>, launch_grid(ceil_div_u(N, kET)), dim3(kET), 0, s, (const c128*)state,
                           (c128*)out, a, acc);
      else
        hipLaunchKernelGGL(k_pauli_apply<float>, launch_grid(ceil_div_u(N, kET)), dim3(kET), 0, s, (const c64*)state,
                           (c64*)out, a, acc);
      QSIM_CHECK_LAUNCH();
    }
    return QSIM_OK;
  }
  if (dtype == QSIM_C128)
    return apply_impl<double>(state, 1, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, nullptr, nullptr, s,
                              "qsim_apply_pauli_sum");
  return apply_impl<float>(state, 1, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, nullptr, nullptr, s,
                           "qsim_apply_pauli_sum");
}

size_t qsim_apply_pauli_sum_batched_workspace(int nbatch, int nterms) {
  if (nbatch < 1 || nterms < 1) return 0;
  return size_t(apply_launches(nterms)) * size_t(nbatch) * kEBlocks * sizeof(double);
}

int qsim_apply_pauli_sum_batched(const void* states, int nbatch, int nqubits, int dtype, int nterms,
                                 const uint64_t* xmasks, const uint64_t* zmasks, const int* ny, const double* coeffs,
                                 void* out, double* energies, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  const char* who = "qsim_apply_pauli_sum_batched";
  QSIM_CHECK_ARG(states != nullptr && out != nullptr && states != out && energies != nullptr && workspace != nullptr,
                 "qsim_apply_pauli_sum_batched: bad pointers");
  QSIM_CHECK_ARG(dtype == QSIM_C128 || dtype == QSIM_C64, "qsim_apply_pauli_sum_batched: bad dtype");
  QSIM_CHECK_ARG(nqubits >= 1 && nqubits <= QSIM_MAX_QUBITS, "qsim_apply_pauli_sum_batched: nqubits out of range");
  QSIM_CHECK_ARG(nbatch >= 1 && nbatch <= 65535, "qsim_apply_pauli_sum_batched: 1..65535 states");
  QSIM_CHECK_ARG(nterms >= 1 && xmasks && zmasks && ny && coeffs, "qsim_apply_pauli_sum_batched: bad term table");
  const uint64_t full = (uint64_t(1) << nqubits) - 1;
  for (int t = 0; t < nterms; ++t)
    QSIM_CHECK_ARG((xmasks[t] & ~full) == 0 && (zmasks[t] & ~full) == 0,
                   "qsim_apply_pauli_sum_batched: mask out of range");
  QSIM_CHECK_ARG(workspace_bytes >= qsim_apply_pauli_sum_batched_workspace(nbatch, nterms),
                 "qsim_apply_pauli_sum_batched: workspace too small");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  double* partial = reinterpret_cast<double*>(workspace);
  if (dtype == QSIM_C128)
    return apply_impl<double>(states, nbatch, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, energies, partial, s,
                              who);
  return apply_impl<float>(states, nbatch, nqubits, nterms, xmasks, zmasks, ny, coeffs, out, energies, partial, s, who);
}

int qsim_inner_matrix(const void* bra, const void* ket, int nqubits, int dtype, const int* targets, int ntargets,
                      const int* controls, int ncontrols, const void* matrix, double* out, void* workspace,
                      size_t workspace_bytes, void* stream) {
  clear_error();
  QSIM_CHECK_ARG(bra && ket && matrix && out && workspace, "qsim_inner_matrix: null pointer");
  QSIM_CHECK_ARG(dtype == QSIM_C128 || dtype == QSIM_C64, "qsim_inner_matrix: bad dtype");
  QSIM_CHECK_ARG(ntargets >= 1 && ntargets <= 3, "qsim_inner_matrix: 1..3 targets supported");
  QSIM_CHECK_ARG(workspace_bytes >= kEBlocks * sizeof(double), "qsim_inner_matrix: workspace too small");
  if (!validate_qubits(nqubits, targets, ntargets, controls, ncontrols, "qsim_inner_matrix")) return QSIM_EINVAL;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  double* partial = reinterpret_cast<double*>(workspace);
  if (dtype == QSIM_C128) {
    switch (ntargets) {
      case 1: return launch_inner<double, 1>(bra, ket, nqubits, targets, controls, ncontrols, matrix, out, partial, s);
      case 2: return launch_inner<double, 2>(bra, ket, nqubits, targets, controls, ncontrols, matrix, out, partial, s);
      default: return launch_inner<double, 3>(bra, ket, nqubits, targets, controls, ncontrols, matrix, out, partial, s);
    }
  }
  switch (ntargets) {
    case 1: return launch_inner<float, 1>(bra, ket, nqubits, targets, controls, ncontrols, matrix, out, partial, s);
    case 2: return launch_inner<float, 2>(bra, ket, nqubits, targets, controls, ncontrols, matrix, out, partial, s);
    default: return launch_inner<float, 3>(bra, ket, nqubits, targets, controls, ncontrols, matrix, out, partial, s);
  }
}

}  // extern "C"
