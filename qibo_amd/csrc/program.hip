// Host-side compiler of one blocked pass into the form the backend runs
// (qsim_compile_program). qsim_compile_pass (compile.hip) keeps the local bits
// in three fixed mappings and is restated record for record in Python; this
// compiler starts from the same planned gates and dependency rules and goes
// further where that is cheaper on the device:
//
//  * any four of the pass's local bits may be register bits (MAP records with
//    layouts): a change of layout picks the bits that let the most waiting
//    gates run, two-qubit gates included, which then run in registers
//    (DENSE2: at most 0.25 CU-cycles per amplitude) instead of through an LDS
//    gather (DENSE_LDS: 0.75);
//  * a SWAP, and the SWAP part of a gate like iSWAP, only renames two local
//    bits: no data moves until the next change of layout;
//  * rotations are divided by their cosines (ROTS: two multiply-adds per real
//    pair instead of three), the cosines multiplied into the entries of records
//    that multiply the whole state at once, a bounded run of rotations each;
//  * a diagonal gate between one register bit and lane bits is split into a
//    table, a per-lane phase and a controlled phase (0.30 CU-cycles as DIAG).
//    Factors of one table or phase are multiplied in extended precision, a
//    lane's diag(a, b) is a factor a of the whole state and b / a on half the
//    lanes, so that an amplitude is rounded no more often than gate by gate;
//  * phases whose conditions lie outside the tile are skipped by whole
//    workgroups; the controlled phases of one register bit share a record;
//  * X gates without a condition on a lane bit exchange registers.

#include <algorithm>
#include <array>
#include <deque>

#include "compile_ops.h"

namespace {

constexpr uint8_t kRRotS = 13, kRDense2 = 14, kRFlip = 15, kRLrpMany = 16;
constexpr int kMaxPhases = 48;  // of one LRPMANY record
constexpr int kMapLayout = 3, kMapStart = 4, kMapRelabel = 5;

// Local bits of one kind share the low bits of their LDS slot (blocked_dev.h:
// swl, kSlotW): the first five lane positions take bits of five kinds.
constexpr int kBankKind[kTileBits] = {0, 1, 2, 3, 4, 0, 1, 2, 4, 3, 0, 1};

// Factors that the compiler multiplies together are kept in extended precision
// and rounded where a record takes them: each record then costs an amplitude
// the one rounding of its own product.
struct L {
  long double re, im;

  L() {}  // (not set)
  L(long double r, long double i) : re(r), im(i) {}
  L(const C& c) : re(c.re), im(c.im) {}
  C rounded() const { return {double(re), double(im)}; }
  long double norm2() const { return re * re + im * im; }
  bool one() const { return re == 1 && im == 0; }
};
inline L operator*(const L& a, const L& b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
inline L operator/(const L& a, const L& b) {
  const long double m = b.norm2();
  return a * L{b.re / m, -b.im / m};
}

struct Item {
  Op op;
  uint32_t need = 0;   // local bits that must be register bits
  bool lds = false;    // runs through LDS in any layout (last choice)
  bool relabel = false;
  int weight = 0;      // gates it counts for when a layout is chosen
};

struct Layout {
  uint8_t at[kTileBits];  // local bit at each position (0-7 lane, 8-11 register)

  uint32_t regs() const {
    uint32_t m = 0;
    for (int p = 8; p < kTileBits; ++p) m |= 1u << at[p];
    return m;
  }
  uint64_t word() const {
    uint64_t w = 0;
    for (int p = 0; p < kTileBits; ++p) w |= uint64_t(at[p]) << (4 * p);
    return w;
  }
  int reg_of(int lb) const {
    for (int p = 8; p < kTileBits; ++p)
      if (at[p] == lb) return p - 8;
    return -1;
  }
};

// The layout with the register bits R: the pass's lowest bits at the lowest
// lane positions (whole lines per access of a lane group), then bits of the
// kinds the first five positions still lack, then the rest ascending.
Layout make_layout(uint32_t R, int low) {
  Layout l;
  int p = 0;
  uint32_t left = ((1u << kTileBits) - 1) & ~R, kinds = 0;
  auto take = [&](int b) {
    l.at[p++] = uint8_t(b);
    left &= ~(1u << b);
    kinds |= 1u << kBankKind[b];
  };
  for (int b = 0; b < low; ++b)
    if ((left >> b) & 1) take(b);
  while (p < 5) {
    int pick = -1;
    for (int b = 0; b < kTileBits && pick < 0; ++b)
      if (((left >> b) & 1) && !((kinds >> kBankKind[b]) & 1)) pick = b;
    if (pick < 0) pick = __builtin_ctz(left);  // a kind held by the registers alone: two lanes share a bank
    take(pick);
  }
  while (left) take(__builtin_ctz(left));
  for (int b = 0; b < kTileBits; ++b)
    if ((R >> b) & 1) l.at[p++] = uint8_t(b);
  return l;
}

// LDS slot of a local index in the interpreter's exchanges (swl in
// blocked_dev.h: linear, so the slots of single bits are combined by XOR).
uint32_t slot_of(uint32_t u, int itemsize) {
  uint32_t s = u ^ ((u >> 5) & 7u) ^ (((u >> 8) & 1u) << 4) ^ (((u >> 9) & 1u) << 3) ^ (((u >> 10) & 1u) * 31u) ^
               (((u >> 11) & 1u) * 30u);
  if (itemsize == 8) s ^= uint32_t(__builtin_popcount(u >> 6) & 1) << 5;
  return s * uint32_t(itemsize / 2);
}

class Compiler {
 public:
  Compiler(int n, const int* tile_bits, int low, Writer& w) : n_(n), tb_(tile_bits), low_(low), w_(w) {
    for (int b = 0; b < 64; ++b) local_[b] = -1;
    for (int i = 0; i < kTileBits; ++i) local_[tile_bits[i]] = i;
    lowmask_ = (1u << low) - 1;
  }

  int run(std::vector<Op>& ops, int* switches);

 private:
  int n_;
  const int* tb_;
  int low_;
  uint32_t lowmask_;
  Writer& w_;
  int local_[64];
  std::vector<Item> items_;
  std::deque<std::array<C, 16>> made_;  // entries of gates rewritten here
  std::vector<std::vector<int>> succ_;
  std::vector<int> npred_, ready_;

  Layout lay_;
  bool stale_ = false;  // lane positions were renamed since the kernel formed the lane's index
  bool relabelled_unseen_ = false;  // any position was renamed since the kernel last saw a layout
  bool have_pending_ = false;  // diagonal gates on the registers not emitted yet:
  L bit_[4][2];                // factors of single register bits, and if `mixed_`
  bool mixed_ = false;
  L pending_[16];              // a table of the others
  long reg_first_off_ = -1;
  size_t reg_first_ev_ = 0;
  L gfac_{1, 0};  // a factor of the whole state, taken by the first record that can
  bool sign_ = false;
  int qpend_ = -1;
  std::vector<std::pair<int, L>> phases_;  // controlled phases of register qpend_ not emitted yet: (bit, phase)
  int switches_ = 0;

  // rotations and the records that can take their cosines, in order
  struct Event {
    int kind;  // 0 rotation, 1 takes factors, 2 a table of some registers
    long off;  // rotation: header; others: first entry
    double t = 0, s = 0, tan = 0, c = 0;
    int dep = 0;
    std::vector<L> entries;
  };
  std::vector<Event> events_;

  void note(uint8_t op, int arg, uint64_t cmask, uint64_t tmask, int rreq, const C* data, int ndata);
  void emit(uint8_t op, int arg, uint64_t cmask, int nt, const int* bits, int nbits, const C* data, int ndata,
            int rreq = 0, uint64_t tmask = 0, bool lane_index = false);
  void build_items(std::vector<Op>& ops);
  void dependencies();
  uint32_t choose_regs(bool first);
  void change_layout(uint32_t R);
  void flush_reg(int j);
  void qflush(int j);
  void emit_phases();
  void emit_diag(const Op& o);
  void emit_table(int dep, const L* table);
  void rewrite(Event& e);
  void emit_phase(const int* tbits, int nt, const int* cbits, int nc, const L* d);
  void emit_dense1(const Op& o, int j);
  void emit_dense2(const Op& o);
  void emit_lds(const Op& o);
  void fold_cosines();
  int gbit(int lb) const { return tb_[lb]; }
  uint64_t outside(uint64_t m) const {
    uint64_t o = 0;
    for (int b = 0; b < 64; ++b)
      if (((m >> b) & 1) && local_[b] < 0) o |= uint64_t(1) << b;
    return o;
  }
};

// Remembers a record that multiplies the whole state, or a table of some
// registers, as a place for the cosines. (Not LANE_PHASE: it multiplies the
// lane's pending factor, which would gather the cosines of several runs of
// rotations while the state already holds their secants: complex64 RX(pi)
// four times beside RZ ended as inf * 0.)
void Compiler::note(uint8_t op, int arg, uint64_t cmask, uint64_t tmask, int rreq, const C* data, int ndata) {
  if (cmask || tmask || rreq || !data) return;
  Event e;
  e.off = long(w_.len) + kHeader;
  if (op != kRRegPhase) e.entries.assign(data, data + ndata);  // (a table's: emit_table)
  if (op == kRRegPhase && arg != 0) {
    e.kind = 2;
    e.dep = arg;
  } else if (op == kRDense1 || op == kRDense1Real || op == kRRegPhase || op == kRDiag || op == kRDense2) {
    e.kind = 1;
  } else {
    return;
  }
  events_.push_back(std::move(e));
}

void Compiler::emit(uint8_t op, int arg, uint64_t cmask, int nt, const int* bits, int nbits, const C* data, int ndata,
                    int rreq, uint64_t tmask, bool lane_index) {
  if (stale_ && (cmask != 0 || lane_index)) {
    stale_ = relabelled_unseen_ = false;
    w_.emit(kRMap, kMapRelabel, lay_.word(), 0, nullptr, 0, nullptr, 0);
  }
  note(op, arg, cmask, tmask, rreq, data, ndata);
  const size_t at = w_.len;
  w_.emit(op, arg, cmask, nt, bits, nbits, data, ndata, rreq);
  if (!w_.overflow && tmask) std::memcpy(w_.out + at + 24, &tmask, 8);
}

void Compiler::build_items(std::vector<Op>& ops) {
  for (Op& o : ops) {
    Item it;
    if (o.kind == kDense && o.nt == 2 && o.nc == 0) {
      // one entry per row in the pattern of a SWAP: a SWAP, then a diagonal
      const C* m = o.data;
      auto zero = [&](int i) { return m[i].re == 0 && m[i].im == 0; };
      bool swap = true;
      for (int i = 0; i < 16; ++i) swap = swap && (zero(i) != (i == 0 || i == 6 || i == 9 || i == 15));
      if (swap) {
        Op d = o;
        made_.emplace_back();
        made_.back()[0] = m[0], made_.back()[1] = m[6], made_.back()[2] = m[9], made_.back()[3] = m[15];
        d.kind = kDiag;
        d.data = made_.back().data();
        d.ndata = 4;
        d.nd_mask = 0;
        o.kind = kSwap;
        o.data = nullptr;
        o.ndata = 0;
        it.op = o;
        it.relabel = true;
        items_.push_back(it);
        bool one = true;
        for (int i = 0; i < 4; ++i) one = one && d.data[i].re == 1 && d.data[i].im == 0;
        if (!one) {
          Item id;
          id.op = d;
          items_.push_back(id);
        }
        continue;
      }
    }
    it.op = o;
    if (o.kind == kSwap) {
      it.relabel = o.nc == 0;
      it.lds = o.nc != 0;
    } else if (o.kind == kDense) {
      if (o.nt == 1 || (o.nt == 2 && o.nc == 0)) {
        for (int k = 0; k < o.nt; ++k) it.need |= 1u << local_[n_ - 1 - o.t[k]];
        it.weight = o.nt == 1 ? 1 : 3;
      } else {
        it.lds = true;
      }
    }
    items_.push_back(it);
  }
}

// As qsim_compile_pass: per amplitude bit, a non-diagonal user follows the
// last non-diagonal user and every diagonal user since, a diagonal user the
// last non-diagonal one.
void Compiler::dependencies() {
  const int N = int(items_.size());
  succ_.assign(size_t(N), {});
  npred_.assign(size_t(N), 0);
  int last_nd[64];
  for (int b = 0; b < 64; ++b) last_nd[b] = -1;
  std::vector<int> since[64];
  std::vector<int> preds;
  for (int j = 0; j < N; ++j) {
    const Op& o = items_[size_t(j)].op;
    preds.clear();
    for (uint64_t m = o.all_mask; m; m &= m - 1) {
      const int b = __builtin_ctzll(m);
      const bool nd = (o.nd_mask >> b) & 1;
      if (nd) preds.insert(preds.end(), since[b].begin(), since[b].end());
      if (last_nd[b] >= 0) preds.push_back(last_nd[b]);
      if (nd) {
        last_nd[b] = j;
        since[b].clear();
      } else {
        since[b].push_back(j);
      }
    }
    std::sort(preds.begin(), preds.end());
    preds.erase(std::unique(preds.begin(), preds.end()), preds.end());
    for (int i : preds) succ_[size_t(i)].push_back(j);
    npred_[size_t(j)] = int(preds.size());
  }
  for (int i = 0; i < N; ++i)
    if (npred_[size_t(i)] == 0) ready_.push_back(i);
}

// The register bits of the next layout: grown greedily by the bits of a
// waiting gate that let the most gates run per bit added (every gate that
// then becomes ready and runs counts, renames included).
uint32_t Compiler::choose_regs(bool first) {
  struct Sim {
    std::vector<int> left, blocked;
    uint32_t R = 0;
    int done = 0;
  };
  auto extend = [&](Sim& s, uint32_t add) {
    s.R |= add;
    std::vector<int> work;
    bool again = true;
    while (again) {
      again = false;
      size_t keep = 0;
      for (size_t i = 0; i < s.blocked.size(); ++i) {
        const int g = s.blocked[i];
        const Item& it = items_[size_t(g)];
        if (!it.lds && !(it.need & ~s.R))
          work.push_back(g);
        else
          s.blocked[keep++] = g;
      }
      s.blocked.resize(keep);
      while (!work.empty()) {
        const int g = work.back();
        work.pop_back();
        const Item& it = items_[size_t(g)];
        s.done += it.weight;
        if (it.relabel) {
          const uint32_t a = 1u << local_[n_ - 1 - it.op.t[0]], b = 1u << local_[n_ - 1 - it.op.t[1]];
          const bool ra = s.R & a, rb = s.R & b;
          if (ra != rb) {
            s.R ^= a | b;
            again = true;
          }
        }
        for (int j : succ_[size_t(g)])
          if (--s.left[size_t(j)] == 0) {
            const Item& nx = items_[size_t(j)];
            if (!nx.lds && !(nx.need & ~s.R))
              work.push_back(j);
            else
              s.blocked.push_back(j);
          }
      }
    }
  };
  Sim cur;
  cur.left = npred_;
  cur.blocked = ready_;
  uint32_t chosen = 0;
  extend(cur, 0);
  const uint32_t banned = first ? lowmask_ : 0;
  while (__builtin_popcount(chosen) < 4) {
    uint32_t cands[96];
    int nc = 0;
    auto add_cand = [&](uint32_t m) {
      m &= ~chosen;
      if (!m || (m & banned) || __builtin_popcount(chosen | m) > 4 || nc == 96) return;
      for (int i = 0; i < nc; ++i)
        if (cands[i] == m) return;
      cands[nc++] = m;
    };
    for (int g : cur.blocked)
      if (!items_[size_t(g)].lds) add_cand(items_[size_t(g)].need & ~cur.R);
    uint32_t best = 0;
    double best_score = 0;
    Sim best_sim;
    for (int i = 0; i < nc; ++i) {
      Sim s = cur;
      extend(s, cands[i]);
      const double score = double(s.done - cur.done) / __builtin_popcount(cands[i]);
      if (score > best_score) {
        best_score = score;
        best = cands[i];
        best_sim = std::move(s);
      }
    }
    if (!best) break;
    chosen |= best;
    cur = std::move(best_sim);
  }
  // compile_pass's groups, where one lets more gates run in all (12 qubits of
  // ten RY, RZ and CZ layers: 9 changes instead of 12, 42 tables instead of 54)
  for (int g = 0; g < 3; ++g) {
    uint32_t m = 0;
    for (int j = 0; j < 4; ++j) m |= 1u << kRegGroups[g][j];
    if (m & banned) continue;
    Sim s;
    s.left = npred_;
    s.blocked = ready_;
    extend(s, m);
    if (s.done > cur.done) {
      chosen = m;
      cur = std::move(s);
    }
  }
  // the rest: bits that leave every kind of bank to the lanes, highest first
  for (int pass = 0; pass < 2; ++pass)
    for (int b = kTileBits - 1; b >= 0 && __builtin_popcount(chosen) < 4; --b) {
      if (((chosen >> b) & 1) || ((lowmask_ >> b) & 1)) continue;
      if (pass == 0) {
        uint32_t kinds = 0;
        for (int c = 0; c < kTileBits; ++c)
          if (!((chosen >> c) & 1) && c != b) kinds |= 1u << kBankKind[c];
        if (kinds != 31u) continue;
      }
      chosen |= 1u << b;
    }
  return chosen;
}

void Compiler::change_layout(uint32_t R) {
  flush_reg(-1);
  qflush(-1);
  const Layout to = make_layout(R, low_);
  const uint64_t from = lay_.word();
  int bytes[8];
  for (int i = 0; i < 8; ++i) bytes[i] = int((from >> (8 * i)) & 255);
  // the interpreter's words (lay_remap_words)
  uint32_t words[64];
  auto slot = [&](const Layout& l, int p) { return slot_of(1u << l.at[p], w_.itemsize); };
  for (int p = 0; p < 8; ++p) {
    const uint64_t g = uint64_t(1) << gbit(to.at[p]);
    words[2 * p] = uint32_t(g);
    words[2 * p + 1] = uint32_t(g >> 32);
    words[16 + p] = slot(lay_, p);
    words[24 + p] = slot(to, p);
  }
  for (int r = 0; r < 16; ++r) {
    words[32 + r] = words[48 + r] = 0;
    for (int j = 0; j < 4; ++j)
      if ((r >> j) & 1) words[32 + r] ^= slot(lay_, 8 + j), words[48 + r] ^= slot(to, 8 + j);
  }
  const C none[32] = {};
  const size_t at = w_.len + kHeader;
  w_.emit(kRMap, kMapLayout, to.word(), 0, bytes, 8, none, int(sizeof(words)) / w_.itemsize);
  if (!w_.overflow) std::memcpy(w_.out + at, words, sizeof(words));
  lay_ = to;
  stale_ = relabelled_unseen_ = false;
  ++switches_;
}

// The collected phases of register qpend_, before the lanes' bits change
// names or its factor is applied.
void Compiler::emit_phases() {
  const int k = int(phases_.size());
  if (k == 0) return;
  if (k <= 2) {
    for (const auto& p : phases_) {
      const uint64_t cm = uint64_t(1) << p.first, tm = outside(cm);
      const C x = p.second.rounded();
      emit(kRLaneRegPhase, qpend_, cm & ~tm, 0, nullptr, 0, &x, 1, 0, tm);
    }
  } else {
    C data[64] = {};
    uint8_t bits[kMaxPhases] = {};
    for (int i = 0; i < k; ++i) {
      data[i] = phases_[size_t(i)].second.rounded();
      const int b = phases_[size_t(i)].first;
      bits[i] = uint8_t(local_[b] < 0 ? 0x80 | b : b);
    }
    const int extra = (k + w_.itemsize - 1) / w_.itemsize;
    emit(kRLrpMany, qpend_, 0, k, nullptr, 0, data, k + extra, 0, 0, true);
    if (!w_.overflow) {
      const size_t raw = (size_t(k + extra) * size_t(w_.itemsize) + 15) / 16 * 16;
      std::memcpy(w_.out + w_.len - raw + size_t(k) * size_t(w_.itemsize), bits, size_t(k));
    }
  }
  phases_.clear();
}

void Compiler::qflush(int j) {
  if (qpend_ < 0 || (j >= 0 && j != qpend_)) return;
  emit_phases();
  emit(kRQFlush, qpend_, 0, 0, nullptr, 0, nullptr, 0);
  qpend_ = -1;
}

// The pending table, before a gate on register j that does not commute with
// it (j = -1: whatever it holds). After the first table the value at
// register 0 goes to the first one, and the record multiplies only the
// registers whose bits it depends on.
void Compiler::flush_reg(int j) {
  if (!have_pending_) return;
  C now[16];
  for (int r = 0; r < 16 && mixed_; ++r) now[r] = pending_[r].rounded();
  auto depends_on = [&](int k) {
    if (!ceq(bit_[k][0].rounded(), bit_[k][1].rounded())) return true;
    for (int r = 0; r < 16 && mixed_; ++r)
      if (!((r >> k) & 1) && !ceq(now[r], now[r | (1 << k)])) return true;
    return false;
  };
  if (j >= 0 && !depends_on(j)) return;
  have_pending_ = false;
  L full[16];
  full[0] = {1, 0};
  for (int k = 0; k < 4; ++k)
    for (int r = 0; r < (1 << k); ++r) {
      full[r | (1 << k)] = full[r] * bit_[k][1];
      full[r] = full[r] * bit_[k][0];
    }
  for (int r = 0; r < 16 && mixed_; ++r) full[r] = full[r] * pending_[r];
  const L t0 = full[0];
  if (reg_first_off_ < 0 || std::fabs(double(t0.norm2() - 1)) > 1e-12) {
    if (reg_first_off_ < 0) {
      reg_first_off_ = long(w_.len) + kHeader;
      reg_first_ev_ = events_.size();
    }
    emit_table(0, full);
    return;
  }
  int dep = 0;
  for (int k = 0; k < 4; ++k)
    if (depends_on(k)) dep |= 1 << k;
  gfac_ = gfac_ * t0;
  if (!dep) return;
  const L inv = L{1, 0} / t0;
  L table[16];
  for (int r = 0; r < 16; ++r)
    table[r] = (r & dep) ? full[r] * inv : L{1, 0};
  emit_table(dep, table);
}

// A REG_PHASE record of the registers whose bits are in `dep` (0: of all).
void Compiler::emit_table(int dep, const L* table) {
  C data[16];
  for (int r = 0; r < 16; ++r) data[r] = table[r].rounded();
  emit(kRRegPhase, dep, 0, 0, nullptr, 0, data, 16);
  events_.back().entries.assign(table, table + 16);
}

void Compiler::rewrite(Event& e) {
  C data[16];
  for (size_t i = 0; i < e.entries.size(); ++i) data[i] = e.entries[i].rounded();
  w_.rewrite(e.off, data, int(e.entries.size()));
}

// A diagonal on the global bits tbits (first = most significant index bit)
// under the bits cbits.
void Compiler::emit_phase(const int* tbits, int nt, const int* cbits, int nc, const L* d) {
  auto reg = [&](int b) { return local_[b] >= 0 ? lay_.reg_of(local_[b]) : -1; };
  int nreg_t = 0, nreg_c = 0, jt = -1;
  for (int k = 0; k < nt; ++k)
    if (reg(tbits[k]) >= 0) ++nreg_t, jt = k;
  for (int k = 0; k < nc; ++k) nreg_c += reg(cbits[k]) >= 0;
  uint64_t cm = 0;
  int rreq = 0;
  for (int k = 0; k < nc; ++k) {
    if (reg(cbits[k]) >= 0)
      rreq |= 1 << reg(cbits[k]);
    else
      cm |= uint64_t(1) << cbits[k];
  }
  auto unit = [](const L& x) { return std::fabs(double(x.norm2() - 1)) <= 1e-6; };
  C rounded[1 << kMaxTargets];
  for (int i = 0; i < (1 << nt); ++i) rounded[i] = d[i].rounded();
  if (nreg_t == 0 && nreg_c == 0) {
    if (nt == 1 && nc == 0 && unit(d[0]) && unit(d[1])) {  // half the lanes are multiplied instead of all
      gfac_ = gfac_ * d[0];
      const L up = d[1] / d[0];
      if (!up.one()) emit_phase(nullptr, 0, tbits, 1, &up);
      return;
    }
    const uint64_t tm = outside(cm);
    emit(kRLanePhase, 0, cm & ~tm, nt, tbits, nt, rounded, 1 << nt, 0, tm, true);
    return;
  }
  if (nreg_t == nt && nreg_c == nc) {
    if (!have_pending_) {
      for (auto& x : bit_) x[0] = x[1] = {1, 0};
      mixed_ = false;
      have_pending_ = true;
    }
    if (nt + nc == 1) {
      const int j = nt == 1 ? reg(tbits[0]) : reg(cbits[0]);
      if (nt == 1) bit_[j][0] = bit_[j][0] * d[0];
      bit_[j][1] = bit_[j][1] * d[nt];
      return;
    }
    if (!mixed_)
      for (L& x : pending_) x = {1, 0};
    mixed_ = true;
    for (int r = 0; r < 16; ++r) {
      if ((r & rreq) != rreq) continue;
      int di = 0;
      for (int k = 0; k < nt; ++k) di = (di << 1) | ((r >> reg(tbits[k])) & 1);
      if (!d[di].one()) pending_[r] = pending_[r] * d[di];
    }
    return;
  }
  if (nt == 0) {
    if (d[0].re == -1 && d[0].im == 0) {
      emit(kRNeg, 0, cm, 0, nullptr, 0, nullptr, 0, rreq);
      return;
    }
    if ((rreq & (rreq - 1)) == 0) {  // one register bit: the lane's factor of its upper half
      const int j = __builtin_ctz(unsigned(rreq));
      if (qpend_ != j) {
        qflush(-1);
        qpend_ = j;
      }
      if ((cm & (cm - 1)) == 0) {  // one condition: collected
        for (auto& p : phases_)
          if (p.first == __builtin_ctzll(cm)) {
            p.second = p.second * d[0];
            return;
          }
        if (int(phases_.size()) == kMaxPhases) emit_phases();
        phases_.emplace_back(__builtin_ctzll(cm), d[0]);
        return;
      }
      const uint64_t tm = outside(cm);
      emit(kRLaneRegPhase, j, cm & ~tm, 0, nullptr, 0, rounded, 1, 0, tm);
      return;
    }
  }
  // one register bit and lane bits: f(0, lanes) f(1, lanes) / f(0, lanes)
  bool units = true;
  for (int i = 0; i < (1 << nt); ++i) units = units && unit(d[i]);
  if (units && nreg_t + nreg_c == 1) {
    auto phase = [&](std::vector<int> c, L x) {  // x where every bit of c is 1
      if (!x.one()) emit_phase(nullptr, 0, c.data(), int(c.size()), &x);
    };
    std::vector<int> cb(cbits, cbits + nc);
    if (nt == 1 && nreg_t == 1) {  // diag(a, b) on the register bit under lane bits
      phase(cb, d[0]);
      cb.push_back(tbits[0]);
      phase(cb, d[1] / d[0]);
      return;
    }
    if (nt == 1 && nreg_c == 1) {  // diag(a, b) on a lane bit, the register bit among the conditions
      phase(cb, d[0]);
      cb.push_back(tbits[0]);
      phase(cb, d[1] / d[0]);
      return;
    }
    if (nt == 2 && nreg_t == 1 && nc == 0) {
      const int jr = jt, jl = 1 - jt;
      auto at = [&](int r, int l) { return d[(r << (1 - jr)) | (l << (1 - jl))]; };
      const L lane[2] = {at(0, 0), at(0, 1)};
      emit_phase(&tbits[jl], 1, nullptr, 0, lane);
      const L up = at(1, 0) / at(0, 0);
      phase({tbits[jr]}, up);
      phase({tbits[jr], tbits[jl]}, at(1, 1) / at(0, 1) / up);
      return;
    }
  }
  int enc[kMaxTargets];
  for (int k = 0; k < nt; ++k) enc[k] = reg(tbits[k]) >= 0 ? int(kRegFlag | uint32_t(reg(tbits[k]))) : tbits[k];
  emit(kRDiag, 0, cm, nt, enc, nt, rounded, 1 << nt, rreq, 0, true);
}

void Compiler::emit_diag(const Op& o) {
  int tb[kMaxTargets], cb[kMaxControls];
  for (int k = 0; k < o.nt; ++k) tb[k] = n_ - 1 - o.t[k];
  for (int k = 0; k < o.nc; ++k) cb[k] = n_ - 1 - o.c[k];
  L d[1 << kMaxTargets];
  std::copy(o.data, o.data + o.ndata, d);
  emit_phase(tb, o.nt, cb, o.nc, d);
}

void Compiler::emit_dense1(const Op& o, int j) {
  flush_reg(j);
  qflush(j);
  uint64_t cm = 0;
  int rreq = 0;
  for (int k = 0; k < o.nc; ++k) {
    const int b = n_ - 1 - o.c[k];
    const int r = local_[b] >= 0 ? lay_.reg_of(local_[b]) : -1;
    if (r >= 0)
      rreq |= 1 << r;
    else
      cm |= uint64_t(1) << b;
  }
  const C* m = o.data;
  int mode;
  double t, s;
  bool neg;
  if (cm == 0 && rreq == 0 && rotation_form(m, w_.itemsize == 16 ? 1e-14 : 4e-7, &mode, &t, &s, &neg)) {
    double c = std::fabs(m[0].re);
    const double norm = std::hypot(c, s);  // (complex64 entries: the rotation by atan2(s, c))
    Event e;
    e.kind = 0;
    e.off = long(w_.len);
    e.t = t;
    e.s = s;
    e.c = c / norm;
    e.tan = c > 0 ? s / c : 0;
    events_.push_back(e);
    w_.emit_rot(j | (mode << 2), t, s);  // fold_cosines turns it into ROTS
    sign_ ^= neg;
    return;
  }
  const bool x = m[0].re == 0 && m[0].im == 0 && m[3].re == 0 && m[3].im == 0 && m[1].re == 1 && m[1].im == 0 &&
                 m[2].re == 1 && m[2].im == 0;
  if (x && cm == 0) {  // a lane condition: 0.17 CU-cycles per amplitude, as DENSE1_REAL 0.10
    emit(kRFlip, j, cm, 0, nullptr, 0, nullptr, 0, rreq);
    return;
  }
  bool real = true;
  for (int k = 0; k < 4 && real; ++k) real = m[k].im == 0;
  emit(real ? kRDense1Real : kRDense1, j, cm, 0, nullptr, 0, m, 4, rreq);
}

void Compiler::emit_dense2(const Op& o) {
  const int j0 = lay_.reg_of(local_[n_ - 1 - o.t[0]]), j1 = lay_.reg_of(local_[n_ - 1 - o.t[1]]);
  flush_reg(j0);
  flush_reg(j1);
  qflush(j0);
  qflush(j1);
  C m[16];
  auto role = [&](int c) { return j0 > j1 ? c : ((c & 1) << 1) | (c >> 1); };
  for (int r = 0; r < 4; ++r)
    for (int c = 0; c < 4; ++c) m[4 * role(r) + role(c)] = o.data[4 * r + c];
  bool real = true, cross = true;
  for (int r = 0; r < 4; ++r)
    for (int c = 0; c < 4; ++c) {
      const C x = m[4 * r + c];
      real = real && x.im == 0;
      if (c != r && c != 3 - r) cross = cross && x.re == 0 && x.im == 0;
    }
  const int hi = std::max(j0, j1), lo = std::min(j0, j1);
  static const int kPair[4][4] = {{-1, -1, -1, -1}, {0, -1, -1, -1}, {1, 3, -1, -1}, {2, 4, 5, -1}};
  const int kind = (cross ? 2 : 0) + (real ? 1 : 0);
  emit(kRDense2, kPair[hi][lo] | (kind << 3), 0, 0, nullptr, 0, m, 16);
}

void Compiler::emit_lds(const Op& o) {
  static const C kSwapMat[16] = {{1, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1, 0}, {0, 0},
                                 {0, 0}, {1, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1, 0}};
  flush_reg(-1);
  qflush(-1);
  const C* mat = o.kind == kSwap ? kSwapMat : o.data;
  const int k = o.nt;
  int bits[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int lb[3] = {0, 0, 0};
  for (int q = 0; q < k; ++q) bits[q] = lb[q] = local_[n_ - 1 - o.t[q]];
  std::sort(lb, lb + k);
  for (int q = 0; q < k; ++q) bits[4 + q] = lb[q];
  uint64_t cm = 0;
  for (int q = 0; q < o.nc; ++q) cm |= uint64_t(1) << (n_ - 1 - o.c[q]);
  // (its amplitudes go through LDS under the layout the kernel holds)
  if (relabelled_unseen_) {
    stale_ = relabelled_unseen_ = false;
    w_.emit(kRMap, kMapRelabel, lay_.word(), 0, nullptr, 0, nullptr, 0);
  }
  w_.emit(kRDenseLds, k, cm, 0, bits, 8, mat, (1 << k) * (1 << k));
}

// Rotations become ROTS records (and the sign of the pass goes to the first
// record that can take it): each cosine goes to the last record before it
// that multiplies the whole state (rotations before the first such record:
// to that one). At most kRunDouble or kRunSingle of them share a record, so
// that the state stays in range between its cosines and its secants; a longer
// run goes on with the next table of some registers, made one of all, or with
// a table of its own where that pays (64 operations against 16 saved per
// rotation). Structure alone decides this, so that a kernel specialised to the
// records serves other angles too: over uniform angles the product of a full
// run's cosines is below the floor once in 10^7 runs or less (the Chernoff
// bound over E |cos|^-0.69 is 9e-8 in complex64, 1e-34 in complex128). Several
// angles near pi in one run pass it: those rotations stay three shears.
constexpr int kRunDouble = 128, kRunSingle = 16, kTablePays = 5;

void Compiler::fold_cosines() {
  const bool single = w_.itemsize == 8;
  const double floor = single ? 0x1p-64 : 0x1p-400;
  const int longest = single ? kRunSingle : kRunDouble;
  const size_t n = events_.size();
  // rotations from each event to the next record that takes cosines or could
  std::vector<int> ahead(n + 1, 0);
  int lead = 0, nrot = 0;  // rotations before the first such record, in all
  bool any = false;
  for (size_t i = n; i-- > 0;) ahead[i] = events_[i].kind == 0 ? ahead[i + 1] + 1 : 0;
  for (const Event& e : events_) {
    nrot += e.kind == 0;
    any = any || e.kind == 1;
    lead += e.kind == 0 && !any;
  }
  if (!any && nrot < kTablePays) {
    if (sign_) w_.emit(kRNeg, 0, 0, 0, nullptr, 0, nullptr, 0);
    return;
  }
  struct Target {
    long off;  // of the added table; -1: the entries of `event`
    size_t event;
    long double factor = 1.0L;
  };
  std::vector<Target> targets;
  int run = 0;
  if (any && lead <= longest) {
    size_t first = 0;
    while (events_[first].kind != 1) ++first;
    targets.push_back({-1, first});
  } else {
    size_t first = 0;
    while (events_[first].kind != 0) ++first;
    targets.push_back({events_[first].off, 0});
    lead = 0;
  }
  for (size_t i = 0; i < n; ++i) {
    Event& e = events_[i];
    if (e.kind == 2 && run + ahead[i + 1] > longest) {
      e.kind = 1;
      w_.out[e.off - kHeader + 1] = 0;  // a table of all registers
    }
    if (e.kind == 1) {
      if (targets.back().off < 0 && targets.back().event == i) continue;  // the lead's: its run goes on
      targets.push_back({-1, i});
      run = 0;
    }
    if (e.kind != 0) continue;
    if (run == longest) {
      if (ahead[i] < kTablePays) continue;
      targets.push_back({e.off, 0});
      run = 0;
    }
    ++run;
    // 1 / sqrt(1 + t^2) of the rounded tangent, multiplied in extended precision:
    // the rotations keep the norm, whatever their number (products of rounded
    // cosines put a 23-qubit circuit of 400 gates 4e-15 off it)
    const double tan = single ? double(float(e.tan)) : e.tan;
    const long double cosine = 1.0L / std::sqrt(1.0L + (long double)(tan) * tan);
    long double& factor = targets.back().factor;
    if (!(e.c > 0) || factor * cosine < floor) continue;  // stays three shears
    factor *= cosine;
    uint8_t* h = w_.out + e.off;
    h[0] = kRRotS;
    std::memset(h + 8, 0, 16);
    if (single) {
      const float t = float(tan);
      std::memcpy(h + 8, &t, 4);
    } else {
      std::memcpy(h + 8, &e.tan, 8);
    }
  }
  if (sign_) targets[0].factor = -targets[0].factor;
  for (size_t k = targets.size(); k-- > 0;) {  // from the end: added tables move what follows them
    const Target& t = targets[k];
    if (t.off < 0) {
      if (t.factor == 1.0L) continue;
      Event& e = events_[t.event];
      for (L& x : e.entries) x.re *= t.factor, x.im *= t.factor;
      rewrite(e);
      continue;
    }
    C table[16];
    for (C& x : table) x = {double(t.factor), 0.0};
    const size_t tail = w_.len;
    w_.emit(kRRegPhase, 0, 0, 0, nullptr, 0, table, 16);
    if (w_.overflow) return;
    std::rotate(w_.out + t.off, w_.out + tail, w_.out + w_.len);
  }
}

int Compiler::run(std::vector<Op>& ops, int* switches) {
  events_.reserve(ops.size() + 16);
  build_items(ops);
  dependencies();
  lay_ = make_layout(choose_regs(true), low_);
  w_.emit(kRMap, kMapStart, lay_.word(), 0, nullptr, 0, nullptr, 0);
  auto runs_here = [&](int i, uint32_t R) {
    const Item& it = items_[size_t(i)];
    return !it.lds && !(it.need & ~R);
  };
  while (!ready_.empty()) {
    std::sort(ready_.begin(), ready_.end());
    uint32_t R = lay_.regs();
    int pick = -1;
    for (int i : ready_)
      if (runs_here(i, R)) {
        pick = i;
        break;
      }
    if (pick < 0) {
      bool reg = false;
      for (int i : ready_) reg = reg || !items_[size_t(i)].lds;
      if (reg) {
        const uint32_t next = choose_regs(false);
        change_layout(next);
        for (int i : ready_)
          if (runs_here(i, next)) {
            pick = i;
            break;
          }
        if (pick < 0) return -1;  // cannot happen: the layout runs a waiting gate
      } else {
        pick = ready_[0];
      }
    }
    ready_.erase(std::find(ready_.begin(), ready_.end(), pick));
    for (int j : succ_[size_t(pick)])
      if (--npred_[size_t(j)] == 0) ready_.push_back(j);
    const Item& it = items_[size_t(pick)];
    const Op& o = it.op;
    if (it.relabel) {
      emit_phases();  // (they name bits, which are about to change places)
      const int a = local_[n_ - 1 - o.t[0]], b = local_[n_ - 1 - o.t[1]];
      for (int p = 0; p < kTileBits; ++p) {
        if (lay_.at[p] == a)
          lay_.at[p] = uint8_t(b);
        else if (lay_.at[p] == b)
          lay_.at[p] = uint8_t(a);
        else
          continue;
        if (p < 8) stale_ = true;
      }
      relabelled_unseen_ = true;
    } else if (it.lds) {
      emit_lds(o);
    } else if (o.kind == kDiag) {
      emit_diag(o);
    } else if (o.nt == 1) {
      emit_dense1(o, lay_.reg_of(local_[n_ - 1 - o.t[0]]));
    } else {
      emit_dense2(o);
    }
  }
  flush_reg(-1);
  qflush(-1);
  // the tile is stored in whole lines: no low bit may sit in a register
  if (lay_.regs() & lowmask_) {
    uint32_t R = lay_.regs() & ~lowmask_;
    for (int b = kTileBits - 1; b >= 0 && __builtin_popcount(R) < 4; --b)
      if (!((R >> b) & 1) && !((lowmask_ >> b) & 1)) R |= 1u << b;
    change_layout(R);
  } else if (relabelled_unseen_) {
    w_.emit(kRMap, kMapRelabel, lay_.word(), 0, nullptr, 0, nullptr, 0);
  }
  if (w_.overflow) return 0;
  if (!gfac_.one()) {
    Event* to = reg_first_off_ >= 0 ? &events_[reg_first_ev_] : nullptr;
    for (Event& e : events_)
      if (!to && e.kind == 1) to = &e;
    if (to) {
      for (L& x : to->entries) x = x * gfac_;
      rewrite(*to);
    } else {
      const C x = gfac_.rounded();
      emit(kRLanePhase, 0, 0, 0, nullptr, 0, &x, 1);
    }
  }
  if (w_.overflow) return 0;
  fold_cosines();
  *switches = switches_;
  return 0;
}

}  // namespace

extern "C" {

size_t qsim_compile_program_capacity(int nops, int dtype) {
  if (nops < 0) return 0;
  const size_t item = dtype == QSIM_C64 ? 8 : 16;
  // per op at most a layout change, a rename, table and factor flushes, three
  // records of a split diagonal and its own record (<= 64 entries)
  const size_t per_op = 12 * kHeader + (16 + 16 + 64) * item + 256 + 64;
  return size_t(nops) * 2 * per_op + 16 * kHeader + 64 * item + 2 * 256;
}

int qsim_compile_program(int nqubits, const int* tile_bits, int nops, const int* op_desc, const double* op_data,
                         const int64_t* data_offsets, int dtype, int low_bits, uint8_t* out, size_t capacity,
                         size_t* out_bytes, int* count, int* switches) {
  qsim::clear_error();
  QSIM_CHECK_ARG(nqubits >= kTileBits && nqubits <= QSIM_MAX_QUBITS, "qsim_compile_program: nqubits out of range");
  QSIM_CHECK_ARG(tile_bits != nullptr && out_bytes != nullptr && count != nullptr && switches != nullptr,
                 "qsim_compile_program: null pointer");
  QSIM_CHECK_ARG(nops >= 0 && (nops == 0 || (op_desc && op_data && data_offsets)), "qsim_compile_program: bad ops");
  QSIM_CHECK_ARG(dtype == QSIM_C128 || dtype == QSIM_C64, "qsim_compile_program: bad dtype");
  QSIM_CHECK_ARG(low_bits >= 0 && low_bits < kTileBits, "qsim_compile_program: bad low bits");
  QSIM_CHECK_ARG(out != nullptr && capacity >= qsim_compile_program_capacity(nops, dtype),
                 "qsim_compile_program: output buffer smaller than qsim_compile_program_capacity");
  std::vector<Op> ops;
  if (parse_ops(nqubits, tile_bits, nops, op_desc, op_data, data_offsets, ops, "qsim_compile_program") != QSIM_OK)
    return QSIM_EINVAL;
  Writer w;
  w.out = out;
  w.cap = capacity;
  w.itemsize = dtype == QSIM_C64 ? 8 : 16;
  // bits kept out of the registers at load and store: the low index bits the
  // tile holds in place (at least the 3 the kernels keep whole lines of, at
  // most 8: four bits are left to the registers)
  int low = 0;
  while (low < kTileBits && tile_bits[low] == low && low < std::max(3, std::min(low_bits, 8))) ++low;
  low = std::max(low, 3);
  int sw = 0;
  Compiler c(nqubits, tile_bits, low, w);
  if (c.run(ops, &sw) != 0) {
    qsim::set_error("qsim_compile_program: scheduling failed");
    return QSIM_EINVAL;
  }
  QSIM_CHECK_ARG(!w.overflow, "qsim_compile_program: output buffer overflow");
  *out_bytes = w.len;
  *count = w.count;
  *switches = sw;
  return QSIM_OK;
}

}  // extern "C"
