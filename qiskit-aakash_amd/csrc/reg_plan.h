// reg_plan.h -- host planning of the register-resident tile passes: records of
// a tile's operations, the stages of a register program, blocks of runs of
// single operations.  Plain C++ (no device code); included by dmsim.hip.
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "dmsim.h"

namespace {

// Tile operations (see the tile program kernels for what each kind does).
enum { TOP_1Q = 1, TOP_CX = 2, TOP_2Q = 3, TOP_DENSE = 4, TOP_STAGE = 6, TOP_1QU = 7 };

struct TileOp {
  int32_t kind, k, d[4], param;
  // Swizzled passes: the order in which a thread's group index g enumerates
  // the tile digits the operation leaves free (3 bits per digit, first digit
  // in bits 0-2); the first ones cover distinct bank fields (lds_swz).
  int32_t lanes;
  // FP32 stages on digits >= 1 with 8-byte LDS accesses along digit 0: the
  // order of the free digits other than digit 0, the first two covering the
  // bank fields of LDS index bits 2-3 and 4-5.
  int32_t qlanes;
};

constexpr int kRegTile = 7;   // digits of a register-resident tile
constexpr int kRegVals = 16;  // values of one member (unused ones zero)

// Members of a stage.  A slot is a register digit (0, 1, 2).
enum {
  RM_U1 = 0,    // + slot: unital single-qubit map, 9 values (3x3, rows X Y Z)
  RM_A1 = 3,    // + slot: general single-qubit map, 12 values (rows X Y Z, columns I X Y Z)
  RM_CX = 6,    // + pair: CX, no values; pairs (control, target) (0,1) (1,0) (0,2) (2,0) (1,2) (2,1)
  RM_D1 = 12,   // + slot: scale components X, Y, Z by 3 values
  RM_D2 = 15,   // + pair of slots (0,1) (0,2) (1,2): 16 scales, index 4 i_first + i_second
  RM_CXD = 18,  // + pair as RM_CX: CX, then 16 scales, index 4 i_control + i_target
};

struct RegStage {
  uint32_t nm, mem;       // members: count, first one
  // redistribution into this stage (unused in the first): the slot whose
  // digit is a register digit before and after (it orders the phases), and
  // the LDS offset (coefficients) of one unit of each other digit, for the
  // writer's layout (the previous stage) and the reader's (this stage); a
  // coefficient's offset is the XOR of its digits times their offsets
  uint32_t slot;
  uint32_t wr[3], wl[3], ww;
  uint32_t rr[3], rl[3], rw;
  uint32_t pad[3];
};

// V: double for the operations in their given order, long double where maps
// are composed: a composed map is rounded once, so that its pass rounds less
// than the operations one by one (24 circuits of 2-6 qubits, 50-250 gates,
// noise after each: relative error 5.7e-16 on average, 1.09e-15 one by one,
// 1.20e-15 with maps composed in doubles).
template <typename V>
struct RegItem {
  uint32_t mask;       // tile digits
  int kind;            // 0: single-qubit map, 1: CX, 2: pair scale
  bool scaled;         // CX with 16 pair scales
  bool exact;          // rounds nothing (a CX permutation)
  int d0, d1;
  V v[16];             // rows X, Y, Z (12 values), or 16 pair scales
};

// Kind and values of a single-qubit map: identity (no member), diagonal,
// unital or general.
inline int reg_1q_kind(const double *r) {
  bool unital = true, diag = true, ident = true;
  for (int i = 0; i < 3; ++i) {
    if (r[4 * i] != 0.0) unital = false;
    for (int j = 0; j < 3; ++j) {
      const double x = r[4 * i + 1 + j];
      if (i != j && x != 0.0) diag = false;
      if (x != (i == j ? 1.0 : 0.0)) ident = false;
    }
  }
  if (!unital) return RM_A1;
  return ident ? -1 : diag ? RM_D1 : RM_U1;
}

// The operations of a pass in their given order, one item each (two for a
// scaled CX: the permutation and the scale).
inline std::vector<RegItem<double>> reg_items_in_order(const std::vector<TileOp> &ops,
                                                       const std::vector<double> &vals) {
  std::vector<RegItem<double>> out;
  out.reserve(2 * ops.size());
  for (const TileOp &op : ops) {
    const double *v = vals.data() + op.param;
    RegItem<double> it;
    it.scaled = false;
    it.d0 = op.d[0];
    if (op.kind == TOP_1Q || op.kind == TOP_1QU) {
      it.kind = 0;
      it.d1 = op.d[0];
      it.mask = 1u << op.d[0];
      it.exact = false;
      memcpy(it.v, v, 12 * sizeof(double));
      out.push_back(it);
      continue;
    }
    it.kind = 1;
    it.d1 = op.d[1];
    it.mask = (1u << it.d0) | (1u << it.d1);
    it.exact = true;
    out.push_back(it);
    bool scaled = false;
    for (int i = 1; op.k && i < 16; ++i) scaled = scaled || v[i] != 1.0;
    if (scaled) {
      it.kind = 2;
      it.exact = false;
      memcpy(it.v, v, 16 * sizeof(double));
      out.push_back(it);
    }
  }
  return out;
}

// The map v after e, both rows X, Y, Z of (I, X, Y, Z), into e.
template <typename S>
inline void compose_1q(const S *v, long double *e) {
  long double w[12];
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 4; ++j) {
      long double acc = j == 0 ? (long double)v[4 * i] : 0.0L;
      for (int k = 0; k < 3; ++k) acc += (long double)v[4 * i + 1 + k] * e[4 * k + j];
      w[4 * i + j] = acc;
    }
  memcpy(e, w, sizeof(w));
}

// The pass's operations as register-stage items, free to be reordered where
// they commute: runs of single-qubit maps on one digit become one map, and
// the separable scale of a CX (a depolarising channel on each of its qubits)
// goes into the next map on either digit where one follows before another
// CX, so that the CX itself only permutes registers; what is left stays as a
// scale of its own.
template <typename S>
inline std::vector<RegItem<long double>> reg_items(const std::vector<TileOp> &ops, const std::vector<S> &vals, int m) {
  using Item = RegItem<long double>;
  std::vector<Item> out;
  out.reserve(ops.size());
  int pend[8];  // item index of the single-qubit map a digit's next one joins, or -1
  for (int d = 0; d < m; ++d) pend[d] = -1;
  bool scales = false;
  for (const TileOp &op : ops) {
    const S *v = vals.data() + op.param;
    if (op.kind == TOP_1Q) {
      const int d = op.d[0];
      if (pend[d] < 0) {
        pend[d] = (int)out.size();
        out.emplace_back();
        Item &it = out.back();
        it.mask = 1u << d;
        it.kind = 0;
        it.scaled = it.exact = false;
        it.d0 = it.d1 = d;
        std::copy(v, v + 12, it.v);
      } else {
        compose_1q(v, out[pend[d]].v);
      }
    } else {
      out.emplace_back();
      Item &it = out.back();
      it.d0 = op.d[0];
      it.d1 = op.d[1];
      it.mask = (1u << it.d0) | (1u << it.d1);
      it.kind = 1;
      it.scaled = op.k != 0;
      it.exact = false;
      if (op.k) std::copy(v, v + 16, it.v);
      scales = scales || it.scaled;
      pend[it.d0] = pend[it.d1] = -1;
    }
  }
  if (!scales) return out;
  // scales
  std::vector<Item> res;
  res.reserve(out.size() + 8);
  for (size_t i = 0; i < out.size(); ++i) {
    const Item it = out[i];
    if (it.kind != 1 || !it.scaled) {
      res.push_back(it);
      continue;
    }
    bool scaled = false, separable = it.v[0] == 1.0;
    for (int c = 0; c < 4; ++c)
      for (int t = 0; t < 4; ++t) {
        const double s = (double)it.v[4 * c + t];
        if (s != 1.0 && (c | t)) scaled = true;
        if (!(fabs(s - (double)it.v[4 * c] * (double)it.v[t]) <= 4e-16 * fabs(s))) separable = false;
      }
    Item cx = it;
    cx.scaled = false;
    res.push_back(cx);
    if (!scaled) continue;
    Item *next[2] = {nullptr, nullptr};
    if (separable)
      for (int s = 0; s < 2; ++s) {
        const uint32_t bit = 1u << (s ? it.d1 : it.d0);
        for (size_t j = i + 1; j < out.size(); ++j)
          if (out[j].mask & bit) {
            if (out[j].kind == 0) next[s] = &out[j];
            break;
          }
      }
    for (int s = 0; s < 2; ++s)
      if (next[s])
        for (int r = 0; r < 3; ++r)
          for (int c = 1; c < 4; ++c) next[s]->v[4 * r + c] *= s ? it.v[c] : it.v[4 * c];
    if (next[0] && next[1]) continue;
    Item d = it;
    if (!next[0] && !next[1]) {
      d.kind = 2;
    } else {
      const int s = next[0] ? 1 : 0;
      d.kind = 0;
      d.d0 = d.d1 = s ? it.d1 : it.d0;
      d.mask = 1u << d.d0;
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 4; ++c) d.v[4 * r + c] = c == r + 1 ? (s ? it.v[c] : it.v[4 * c]) : 0.0;
    }
    res.push_back(d);
  }
  return res;
}

// The pending items of a pass or run: each digit has the list of the items
// that touch it, in program order, and so have the items that round
// something.  A stage's items are found by walking the lists of its digits,
// so that planning takes time in proportion to the items taken and not to
// those still pending.
class RegQueue {
 public:
  static constexpr int kEnd = INT32_MAX;

  template <typename V>
  explicit RegQueue(const std::vector<RegItem<V>> &items) : node_(items.size()) {
    for (int &h : head_) h = kEnd;
    for (size_t i = items.size(); i-- > 0;) {
      const RegItem<V> &it = items[i];
      Node &e = node_[i];
      e.mask = it.mask;
      e.list[0] = (int8_t)it.d0;
      e.list[1] = (int8_t)(it.d1 != it.d0 ? it.d1 : -1);
      e.list[2] = (int8_t)(it.exact ? -1 : kRounding);
      ++count_[it.mask];
      for (int s = 0; s < 3; ++s) {
        const int l = e.list[s];
        if (l < 0) continue;
        e.next[s] = head_[l];
        e.prev[s] = kEnd;
        if (head_[l] != kEnd) node_[head_[l]].prev[slot(head_[l], l)] = (int)i;
        head_[l] = (int)i;
      }
    }
  }

  // Pending items inside the triple of digits d.
  int inside(const int (&d)[3]) const {
    int n = 0;
    for (int a = 0; a < 3; ++a) n += count_[1u << d[a]] + count_[(1u << d[a]) | (1u << d[(a + 1) % 3])];
    return n;
  }

  // The digits of the first pending item.
  uint32_t first_mask() const {
    int i = kEnd;
    for (int d = 0; d < kRounding; ++d) i = std::min(i, head_[d]);
    return i == kEnd ? 0u : node_[i].mask;
  }

  // Items that a stage on the digits d takes: an item joins unless it, or an
  // earlier one left out that it does not commute with, reaches outside the
  // triple.  Items on different digits commute; with `ordered` (results bit
  // for bit those of the given order) only if one of them rounds nothing: an
  // item that rounds joins only as the first pending one of those.
  int absorb(const int (&d)[3], bool ordered, std::vector<int> *take) const {
    return take ? (ordered ? walk<true, true>(d, take) : walk<false, true>(d, take))
                : (ordered ? walk<true, false>(d, take) : walk<false, false>(d, take));
  }

  void remove(int i) {
    const Node &e = node_[i];
    --count_[e.mask];
    for (int s = 0; s < 3; ++s) {
      const int l = e.list[s];
      if (l < 0) continue;
      if (e.prev[s] == kEnd) head_[l] = e.next[s];
      else node_[e.prev[s]].next[slot(e.prev[s], l)] = e.next[s];
      if (e.next[s] != kEnd) node_[e.next[s]].prev[slot(e.next[s], l)] = e.prev[s];
    }
  }

 private:
  template <bool ORDERED, bool TAKE>
  int walk(const int (&d)[3], std::vector<int> *take) const {
    const uint32_t triple = (1u << d[0]) | (1u << d[1]) | (1u << d[2]);
    int a = head_[d[0]], b = head_[d[1]], c = head_[d[2]], n = 0;  // next item of each digit, kEnd: blocked or none
    int rounding = ORDERED ? head_[kRounding] : 0;
    uint32_t outside = ~triple;  // and the digits of items left out
    for (;;) {
      const int i = std::min(a, std::min(b, c));
      if (i == kEnd) return n;
      const Node &e = node_[i];
      const bool rounds = ORDERED && e.list[2] >= 0;
      if ((e.mask & outside) || (rounds && i != rounding)) {
        outside |= e.mask;
        if (a == i) a = kEnd;
        if (b == i) b = kEnd;
        if (c == i) c = kEnd;
        continue;
      }
      ++n;
      if (TAKE) take->push_back(i);
      if (rounds) rounding = e.next[2];
      if (a == i) a = e.next[e.list[0] == d[0] ? 0 : 1];
      if (b == i) b = e.next[e.list[0] == d[1] ? 0 : 1];
      if (c == i) c = e.next[e.list[0] == d[2] ? 0 : 1];
    }
  }

  static constexpr int kRounding = 8;  // the list of the items that round
  // An item's lists: its first digit's, its second digit's, the rounding
  // items' (-1: none), and its neighbours in each.
  struct Node {
    uint32_t mask;
    int8_t list[3];
    int next[3], prev[3];
  };
  int slot(int i, int l) const { return l == kRounding ? 2 : node_[i].list[0] == l ? 0 : 1; }

  std::vector<Node> node_;
  int head_[9];
  int count_[256] = {0};  // pending items by digits
};

struct RegLay {
  int r[3], l[3], w, slot;  // register, lane and wave digits, slot that orders the phases
};

struct RegPlan {
  int ns = 0;
  RegLay first, last;           // layouts of the first and the last stage
  std::vector<uint32_t> words;  // RegStage records, then the members' kinds and one spare
  std::vector<double> vals;     // kRegVals values a member, and one spare block
};

// Stages: the first one on a layout that loads HBM directly (register digits
// among 3-6, lanes on digits 0-2: 64 consecutive coefficients per access),
// each further one on the three digits that take the most pending items (at
// least one: an item's digits and one kept from the stage before), and
// a last, possibly empty one on a layout that stores directly.  With
// `ordered` the operations keep their order (see RegQueue::absorb).
// `io`: a tile of a state; otherwise (a whole circuit) any layout may come
// first and last.  m digits (6: no wave digit).
template <typename V>
inline void reg_plan(const std::vector<RegItem<V>> &items, int m, bool io, bool ordered, RegPlan *out) {
  int digits[35][3];
  uint32_t triples[35], nt = 0;
  auto add = [&](int a, int b, int c) {
    digits[nt][0] = a;
    digits[nt][1] = b;
    digits[nt][2] = c;
    triples[nt++] = (1u << a) | (1u << b) | (1u << c);
  };
  for (int a = 3; a < m; ++a)  // the 4 load / store layouts of 7 digits first
    for (int b = a + 1; b < m; ++b)
      for (int c = b + 1; c < m; ++c) add(a, b, c);
  const uint32_t nio = nt;
  for (int a = 0; a < 3; ++a)
    for (int b = a + 1; b < m; ++b)
      for (int c = b + 1; c < m; ++c) add(a, b, c);
  RegQueue queue(items);
  std::vector<uint32_t> stage;
  std::vector<int> order;     // items in the order in which the stages take them
  std::vector<size_t> taken;  // end of each stage's items in `order`
  order.reserve(items.size());
  size_t left = items.size();
  while (left || stage.empty()) {
    const bool load = io && stage.empty();
    const uint32_t first = ordered && !load ? queue.first_mask() : 0u;
    uint32_t best = 0;
    int most = -1;
    for (uint32_t t = 0; t < (load ? nio : nt); ++t) {
      if (!stage.empty() && !(triples[t] & stage.back())) continue;  // a redistribution keeps one digit
      if (first & ~triples[t]) continue;                   // in order, the first pending item comes first
      if (queue.inside(digits[t]) <= most) continue;       // no more than these can be taken
      const int n = queue.absorb(digits[t], ordered, nullptr);
      if (n > most) {
        most = n;
        best = t;
      }
    }
    const size_t from = order.size();
    queue.absorb(digits[best], ordered, &order);
    for (size_t x = from; x < order.size(); ++x) queue.remove(order[x]);
    left -= order.size() - from;
    stage.push_back(triples[best]);
    taken.push_back(order.size());
  }
  if (io && (stage.back() & 7u)) {  // an empty stage that stores directly
    const uint32_t last = stage.back();
    uint32_t best = nio;
    for (uint32_t t = 0; t < nio; ++t)
      if ((triples[t] & last) && (best == nio || __builtin_popcount(triples[t] & last) >
                                                     __builtin_popcount(triples[best] & last)))
        best = t;
    if (best == nio) {  // digits 0-2 in registers: one stage in between
      stage.push_back((1u << 2) | (1u << 3) | (1u << 4));
      taken.push_back(order.size());
      best = 0;  // digits 3, 4, 5
    }
    stage.push_back(triples[best]);
    taken.push_back(order.size());
  }
  const int ns = (int)stage.size();
  std::vector<RegLay> lay(ns);
  for (int k = 0; k < ns; ++k) {
    RegLay &y = lay[k];
    int reg[3], nreg = 0, rest[4], nrest = 0;
    for (int d = 0; d < m; ++d) {
      if ((stage[k] >> d) & 1) reg[nreg++] = d;
      else rest[nrest++] = d;
    }
    // register digits: those kept from the previous stage stay in their
    // slots, the last such slot orders the phases
    for (int j = 0; j < 3; ++j) y.r[j] = -1;
    y.slot = 0;
    if (k) {
      y.slot = -1;
      for (int j = 0; j < 3; ++j)
        if ((stage[k] >> lay[k - 1].r[j]) & 1) {
          y.r[j] = lay[k - 1].r[j];
          y.slot = j;  // the last one
        }
    }
    for (int x = 0; x < 3; ++x) {
      bool held = false;
      for (int j = 0; j < 3; ++j) held = held || y.r[j] == reg[x];
      for (int j = 0; j < 3 && !held; ++j)
        if (y.r[j] < 0) {
          y.r[j] = reg[x];
          held = true;
        }
    }
    // lane digits: digits 0-2 at the lane index of the load / store layouts,
    // digits that were lanes before at their index; the wave digit is the
    // highest of the others
    for (int j = 0; j < 3; ++j) y.l[j] = -1;
    bool used[8] = {false};
    for (int x = 0; x < nrest; ++x)
      if (rest[x] < 3) {
        y.l[rest[x]] = rest[x];
        used[rest[x]] = true;
      }
    if (k)
      for (int j = 0; j < 3; ++j) {
        const int d = lay[k - 1].l[j];
        if (d >= 3 && y.l[j] < 0 && !((stage[k] >> d) & 1)) {
          y.l[j] = d;
          used[d] = true;
        }
      }
    int x = 0;
    for (int j = 0; j < 3; ++j)
      if (y.l[j] < 0) {
        while (used[rest[x]]) ++x;
        y.l[j] = rest[x];
        used[rest[x]] = true;
      }
    y.w = m;  // (no wave digit)
    for (int q = 0; q < nrest; ++q)
      if (!used[rest[q]]) y.w = rest[q];
  }
  out->first = lay[0];
  out->last = lay[ns - 1];
  out->ns = ns;
  out->words.clear();
  out->words.reserve(ns * (sizeof(RegStage) / 4) + items.size() + 1);
  out->vals.clear();
  out->vals.reserve((items.size() + 1) * kRegVals);
  std::vector<uint32_t> kinds;
  kinds.reserve(items.size() + 1);
  for (int k = 0; k < ns; ++k) {
    RegStage sg;
    memset(&sg, 0, sizeof(sg));
    sg.mem = (uint32_t)kinds.size();
    auto slot = [&](int d) { return lay[k].r[0] == d ? 0 : lay[k].r[1] == d ? 1 : 2; };
    for (size_t x = k ? taken[k - 1] : 0; x < taken[k]; ++x) {
      const RegItem<V> &it = items[order[x]];
      double v[kRegVals] = {0.0};
      uint32_t kind;
      if (it.kind == 0) {
        double r12[12];
        for (int c = 0; c < 12; ++c) r12[c] = (double)it.v[c];
        const int k1 = reg_1q_kind(r12);
        if (k1 < 0) continue;
        kind = k1 + slot(it.d0);
        int at = 0;
        for (int r = 0; r < 3; ++r)
          for (int c = 0; c < 4; ++c)
            if (k1 == RM_A1 || (k1 == RM_U1 && c > 0) || (k1 == RM_D1 && c == r + 1)) v[at++] = r12[4 * r + c];
      } else {
        const int s0 = slot(it.d0), s1 = slot(it.d1);
        const int lo = std::min(s0, s1), hi = std::max(s0, s1);
        const int pair = lo == 0 ? hi - 1 : 2;  // (0,1) (0,2) (1,2)
        const RegItem<V> *scale = nullptr;  // the scale of this CX, if it comes next
        if (it.kind == 1 && x + 1 < taken[k]) {
          scale = &items[order[x + 1]];
          if (scale->kind != 2 || scale->d0 != it.d0 || scale->d1 != it.d1) scale = nullptr;
        }
        if (scale) {
          kind = RM_CXD + 2 * pair + (s0 > s1 ? 1 : 0);
          for (int c = 0; c < 16; ++c) v[c] = (double)scale->v[c];
          ++x;
        } else if (it.kind == 1) {
          kind = RM_CX + 2 * pair + (s0 > s1 ? 1 : 0);
        } else {
          kind = RM_D2 + pair;
          for (int a = 0; a < 4; ++a)
            for (int b = 0; b < 4; ++b) v[4 * a + b] = (double)it.v[s0 < s1 ? 4 * a + b : 4 * b + a];
        }
      }
      kinds.push_back(kind);
      out->vals.insert(out->vals.end(), v, v + kRegVals);
    }
    sg.nm = (uint32_t)kinds.size() - sg.mem;
    if (k) {
      // LDS offsets of the digits.  The banks are the lowest three base-4
      // digits of the coefficient index: the writer's lane digits sit there,
      // and a lane digit of the reader that is none of them is added (XOR)
      // to the place of one that is no lane of the reader, so that the lanes of a wave fall on
      // distinct banks on both sides.  Every digit but the writer's lanes
      // and the phase digit also has a place of its own above them.
      const RegLay &w = lay[k - 1], &y = lay[k];
      uint32_t co[8] = {0};
      for (int j = 0; j < 3; ++j) co[w.l[j]] = 1u << (2 * j);
      int high = 3;
      for (int d = 0; d < m; ++d)
        if (!co[d] && d != y.r[y.slot]) co[d] = 1u << (2 * high++);
      bool place[3];  // places of writer lanes that are no reader lanes
      for (int j = 0; j < 3; ++j) place[j] = w.l[j] != y.l[0] && w.l[j] != y.l[1] && w.l[j] != y.l[2];
      for (int j = 0; j < 3; ++j) {
        if (y.l[j] == w.l[0] || y.l[j] == w.l[1] || y.l[j] == w.l[2]) continue;
        int at = j;
        while (!place[at]) at = (at + 1) % 3;
        place[at] = false;
        co[y.l[j]] |= 1u << (2 * at);
      }
      sg.slot = (uint32_t)y.slot;
      for (int j = 0; j < 3; ++j) {
        sg.wr[j] = co[w.r[j]];
        sg.wl[j] = co[w.l[j]];
        sg.rr[j] = co[y.r[j]];
        sg.rl[j] = co[y.l[j]];
      }
      sg.ww = co[w.w];
      sg.rw = co[y.w];
    }
    uint32_t w[sizeof(RegStage) / 4];
    memcpy(w, &sg, sizeof(sg));
    out->words.insert(out->words.end(), w, w + sizeof(RegStage) / 4);
  }
  // the spare member that the last one's prefetch reads
  kinds.push_back(0);
  out->words.insert(out->words.end(), kinds.begin(), kinds.end());
  out->vals.resize(out->vals.size() + kRegVals, 0.0);
}

// Runs of single-qubit, CX and memory-noise operations of a program on an
// FP64 state as fused passes (an FP32 state keeps one kernel per operation:
// its kernels round differently).  Up to 6 qubits, where one kernel takes the
// whole run, the program's own fused passes join it.
// Single-qubit maps of a position with no CX between them are one map; the
// levels of memory noise between two operations of a position join it when
// the second one comes (settle), or at the end of the run (settle_all).
struct PlainRun {
  struct Level {
    long double xy, z, feed;    // factors of X and Y, of Z, and what Z takes from I
    int src;
  };
  std::vector<TileOp> ops;      // digits are positions
  std::vector<long double> vals;
  std::vector<int> src;         // program operation of each (the first one)
  std::vector<int> count;       // operations in each (memory noise: one a position)
  std::vector<Level> levels;
  int pend[32];                 // the map that a position's next one joins, or -1
  int settled[32];              // levels a position has taken
  int total = 0;                // sum of count
  double kernels = 0.0;         // the kernels that run the operations one by one

  PlainRun() {
    for (int p = 0; p < 32; ++p) {
      pend[p] = -1;
      settled[p] = 0;
    }
  }
};

// A map (12 values) or a CX (0 or 16) of `count` operations at the end.
template <typename S>
inline void append_plain(TileOp t, const S *v, int nv, int src, int count, PlainRun *run) {
  t.param = (int32_t)run->vals.size();
  run->vals.insert(run->vals.end(), v, v + nv);
  run->ops.push_back(t);
  run->src.push_back(src);
  run->count.push_back(count);
  run->total += count;
}

inline void settle(int p, PlainRun *run) {
  const int first = run->settled[p], n = (int)run->levels.size() - first;
  if (n == 0) return;
  long double xy = 1.0L, z = 1.0L, feed = 0.0L;
  for (int i = first; i < first + n; ++i) {
    const PlainRun::Level &l = run->levels[i];
    xy *= l.xy;
    z *= l.z;
    feed = l.z * feed + l.feed;
  }
  run->settled[p] = first + n;
  const int at = run->pend[p];
  if (at >= 0) {
    long double *e = &run->vals[run->ops[at].param];
    for (int j = 0; j < 8; ++j) e[j] *= xy;
    for (int j = 8; j < 12; ++j) e[j] *= z;
    e[8] += feed;
    run->count[at] += n;
    run->total += n;
    return;
  }
  const long double R[12] = {0, xy, 0, 0, 0, 0, xy, 0, feed, 0, 0, z};
  TileOp t;
  memset(&t, 0, sizeof(t));
  t.kind = TOP_1Q;
  t.k = 1;
  t.d[0] = p;
  run->pend[p] = (int)run->ops.size();
  append_plain(t, R, 12, run->levels[first].src, n, run);
}

inline void settle_all(int n, PlainRun *run) {
  for (int p = 0; p < n; ++p) settle(p, run);
}

inline bool plain_op(const dm_op &op) {
  return op.kind == DM_OP_1Q || op.kind == DM_OP_CX || op.kind == DM_OP_CX_SCALED || op.kind == DM_OP_MEMORY_NOISE;
}

// One operation (digits are positions) with its nv values; program operation src.
inline void push_plain(TileOp t, const double *v, int nv, int src, PlainRun *run) {
  settle(t.d[0], run);
  if (t.kind == TOP_1Q) {
    int &p = run->pend[t.d[0]];
    if (p >= 0) {
      compose_1q(v, &run->vals[run->ops[p].param]);
      ++run->count[p];
      ++run->total;
      return;
    }
    p = (int)run->ops.size();
  } else {
    settle(t.d[1], run);
    run->pend[t.d[0]] = run->pend[t.d[1]] = -1;
  }
  append_plain(t, v, nv, src, 1, run);
}

// Thermal feed of a memory noise (f, p, g): what its Z component takes from I.
inline double noise_feed(const double *v) { return (1 - v[2]) * (2 * v[1] - 1); }

// The kernels that run one operation by itself, in units of a short launch
// (3-5 us below 12 qubits); a fused pass of a register of up to 6 qubits
// counts 3.  Memory noise is a diagonal kernel or, with a thermal feed, tile
// passes, which at 7-9 qubits take two short launches each (7 qubits, one map
// and one such level: 26 us; two maps 18).
inline double plain_kernels(int n, const dm_op &op, const double *params) {
  if (op.kind == DM_OP_FUSED) return 3;
  if (op.kind != DM_OP_MEMORY_NOISE) return 1;
  const double *v = params + op.param;
  if (v[0] == 1.0 && v[2] == 1.0) return 0;
  if (noise_feed(v) == 0.0) return 1;
  return n >= 12 ? 1 + (n - 4) / 4 : (1 + (n - 4) / 3) * (n >= 7 && n <= 9 ? 2 : 1);
}

// The positions of an operation (a fused pass of a register of up to 6 qubits:
// all), and the fewest blocks of operations on the positions `used`: a block
// takes the positions 0-2 and four others.
inline uint32_t plain_positions(int n, const dm_op &op) {
  if (op.kind == DM_OP_1Q) return 1u << (n - 1 - op.qubits[0]);
  if (op.kind == DM_OP_CX || op.kind == DM_OP_CX_SCALED)
    return (1u << (n - 1 - op.qubits[0])) | (1u << (n - 1 - op.qubits[1]));
  return (1u << n) - 1u;
}
inline size_t least_blocks(uint32_t used) { return std::max(1, (__builtin_popcount(used & ~7u) + 3) / 4); }

// What `blocks` passes instead of the run's own kernels cost, in the same
// units, staging and upload of their image included; the run is fused where
// its kernels cost more.  FP64, one call, us, kernels against passes:
// - up to 6 qubits one launch takes the run: six kernels (5 qubits, 4 maps and
//   4 noise levels 41 against 31; 80 gates in dense blocks with short runs
//   between them 293, and 302 with every run of two and more as one launch);
// - 7-9 qubits: kernels of 4.5 us beside passes of 12-14 and 20 of fixed cost
//   (9 qubits, 4 gates 27 against 34, 8 gates 43 against 35, 4 gates and 4
//   levels, two passes, 42 against 46, 8 and 8 64 against 48);
// - 10 and 11 qubits: kernels of 7-13 us (10 qubits, 4 gates 39 against 35, 4
//   gates and 4 levels 54 against 53);
// - from 12 qubits on a pass takes 1.0-1.4 times a kernel (12 qubits, two
//   gates, one pass, 104 against 58; 13 qubits, 4 gates 700 against 226).
inline double plain_pass_cost(int n, size_t blocks) {
  return n <= 6 ? 5.5 : n <= 9 ? 3.0 * blocks + 3.0 : n <= 11 ? 2.0 * blocks : 1.4 * blocks;
}

inline void add_plain(int n, const dm_op &op, const double *params, int src, PlainRun *run) {
  TileOp t;
  memset(&t, 0, sizeof(t));
  const double *pv = params + op.param;
  run->kernels += plain_kernels(n, op, params);
  if (op.kind == DM_OP_MEMORY_NOISE) {
    const double f = pv[0], g = pv[2];
    if (f != 1.0 || g != 1.0) run->levels.push_back({sqrt(g) * f, g, noise_feed(pv), src});
    return;
  }
  t.d[0] = n - 1 - op.qubits[0];
  if (op.kind == DM_OP_1Q) {
    t.kind = TOP_1Q;
    t.k = 1;
    push_plain(t, pv, 12, src, run);
  } else {
    t.kind = TOP_CX;
    t.d[1] = n - 1 - op.qubits[1];
    t.k = op.kind == DM_OP_CX_SCALED ? 1 : 0;
    push_plain(t, pv, t.k ? 16 : 0, src, run);
  }
}

// Blocks of the run: the operations that the tile of the positions 0-2 and
// up to four others takes (an operation joins unless it, or an earlier one
// left out that shares a position with it, reaches outside), the others
// chosen by growth from the first pending operation, with and without one
// position forced in, whichever takes the most operations.
// Each position has the list of its pending operations, and a block is found
// by walking the lists of the positions still open to it: the time goes with
// the operations taken and not with those left pending.
inline std::vector<std::vector<int>> plain_blocks(int n, const PlainRun &run) {
  constexpr int kEnd = INT32_MAX;
  struct Link {
    int next, prev;
  };
  const int no = (int)run.ops.size();
  std::vector<uint32_t> mask(no);
  std::vector<Link> link(2 * (size_t)no);
  int head[32];
  for (int &h : head) h = kEnd;
  auto at = [&](int i, int p) -> Link & { return link[2 * (size_t)i + (run.ops[i].d[0] == p ? 0 : 1)]; };
  for (int i = no - 1; i >= 0; --i)
    for (int x = 0; x < (run.ops[i].kind == TOP_CX ? 2 : 1); ++x) {
      const int p = run.ops[i].d[x];
      mask[i] |= 1u << p;
      at(i, p) = {head[p], kEnd};
      if (head[p] != kEnd) at(head[p], p).prev = i;
      head[p] = i;
    }
  const uint32_t low = 7u, full = (1u << n) - 1u;
  const int most_high = std::min(4, n - 3);
  std::vector<std::vector<int>> out;
  std::vector<int> cur, best;
  for (int left = no; left;) {
    best.clear();
    int most = 0;
    uint32_t grown = 0;  // the positions of the growth without a forced one: with one of them forced it is the same
    for (int force = -1; force < n; ++force) {
      if (force >= 0 && (((low | grown) >> force) & 1)) continue;
      uint32_t T = force < 0 ? 0 : 1u << force, blocked = 0;
      int walk[32], ops = 0;
      memcpy(walk, head, sizeof(walk));
      cur.clear();
      for (;;) {
        const uint32_t open = (__builtin_popcount(T) < most_high ? full : T | low) & ~blocked;
        int i = kEnd;
        for (uint32_t s = open; s; s &= s - 1) i = std::min(i, walk[__builtin_ctz(s)]);
        if (i == kEnd) break;
        const uint32_t m = mask[i], t2 = T | (m & ~low);
        if ((m & blocked) || __builtin_popcount(t2) > most_high) {
          blocked |= m;
          continue;
        }
        T = t2;
        cur.push_back(i);
        ops += run.count[i];
        for (uint32_t s = m; s; s &= s - 1) {
          const int p = __builtin_ctz(s);
          walk[p] = at(i, p).next;
        }
      }
      if (force < 0) grown = T;
      if (ops > most) {
        most = ops;
        best.swap(cur);
      }
    }
    for (int i : best)
      for (uint32_t s = mask[i]; s; s &= s - 1) {
        const int p = __builtin_ctz(s);
        const Link k = at(i, p);
        if (k.prev == kEnd) head[p] = k.next;
        else at(k.prev, p).next = k.next;
        if (k.next != kEnd) at(k.next, p).prev = k.prev;
      }
    left -= (int)best.size();
    out.push_back(best);
  }
  return out;
}

}  // namespace
