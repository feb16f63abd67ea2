"""Host planning of the register-resident passes (csrc/reg_plan.h), on the CPU.

reg_plan.h is plain C++ and is compiled here with g++ into two drivers:

* what a stage takes and how a run of single operations splits into blocks,
  on random programs, against the definition: walk every pending operation
  in order, an operation joins unless it, or an earlier one left out that it
  does not commute with, reaches outside;
* programs of 400,000 gates whose last digit is never used, or only by the
  last gate: planning time goes with the length of the program.  A planner
  that looks at what is still pending at every stage needs 1e10 steps and
  more (over a minute); the limit of 20 s is some 40 times what it takes;
* maps composed on the host are rounded once, against 113 bits;
* the choice between one kernel an operation and fused passes, at sizes where
  both were timed.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COMMON = r'''
#include <stdio.h>
#include <stdlib.h>
#include <chrono>
#include <random>
#include "reg_plan.h"

static std::mt19937_64 rng(3);
static int uni(int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); }
static const double kOnes[16] = {1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1};
static const double kScale[16] = {1, .9, .9, .9, .9, .8, .8, .8, .9, .8, .8, .8, .9, .8, .8, .8};
static const double kMap[12] = {0, .6, .8, 0, 0, -.8, .6, 0, .1, 0, 0, .9};
'''

DEFINITION = COMMON + r'''
template <typename V>
static std::vector<int> takes(const std::vector<RegItem<V>> &items, const std::vector<char> &done, uint32_t triple,
                              bool ordered) {
  std::vector<int> out;
  uint32_t blocked = 0;
  bool rounded = false;
  for (size_t i = 0; i < items.size(); ++i) {
    if (done[i]) continue;
    const uint32_t m = items[i].mask;
    if ((m & blocked) || (m & ~triple) || (ordered && rounded && !items[i].exact)) {
      blocked |= m;
      rounded = rounded || !items[i].exact;
    } else {
      out.push_back((int)i);
    }
  }
  return out;
}

// Stages on random digits until every item is taken.
template <typename V>
static int walk(const std::vector<RegItem<V>> &items, int m, bool ordered) {
  int bad = 0;
  std::vector<char> done(items.size(), 0);
  RegQueue queue(items);
  size_t left = items.size();
  for (int step = 0; left && step < 10000; ++step) {
    int d[3] = {uni(0, m - 1), 0, 0};
    do d[1] = uni(0, m - 1);
    while (d[1] == d[0]);
    do d[2] = uni(0, m - 1);
    while (d[2] == d[0] || d[2] == d[1]);
    std::sort(d, d + 3);
    const uint32_t triple = (1u << d[0]) | (1u << d[1]) | (1u << d[2]);
    std::vector<int> got;
    const int n = queue.absorb(d, ordered, &got);
    const std::vector<int> want = takes(items, done, triple, ordered);
    int inside = 0, first = -1;
    for (size_t i = 0; i < items.size(); ++i)
      if (!done[i]) {
        inside += (items[i].mask & ~triple) == 0;
        if (first < 0) first = (int)i;
      }
    if (got != want || n != (int)want.size() || queue.inside(d) != inside || queue.first_mask() != items[first].mask)
      ++bad;
    for (int i : want) {
      done[i] = 1;
      queue.remove(i);
    }
    left -= want.size();
  }
  return bad + (left != 0);
}

static int stages() {
  int bad = 0;
  for (int trial = 0; trial < 2000; ++trial) {
    const int m = uni(6, 7), digits = uni(2, m), nops = uni(0, 40);
    const bool ordered = uni(0, 1);
    std::vector<TileOp> ops;
    std::vector<double> vals;
    for (int i = 0; i < nops; ++i) {
      TileOp op;
      memset(&op, 0, sizeof(op));
      op.param = (int32_t)vals.size();
      op.d[0] = uni(0, digits - 1);
      op.kind = uni(0, 1) ? TOP_1Q : TOP_CX;
      if (op.kind == TOP_1Q) {
        vals.insert(vals.end(), kMap, kMap + 12);
      } else {
        do op.d[1] = uni(0, digits - 1);
        while (op.d[1] == op.d[0]);
        op.k = uni(0, 1);
        const double *s = uni(0, 1) ? kScale : kOnes;
        vals.insert(vals.end(), s, s + 16);
      }
      ops.push_back(op);
    }
    bad += ordered ? walk(reg_items_in_order(ops, vals), m, true) : walk(reg_items(ops, vals, m), m, false);
  }
  return bad;
}

static std::vector<std::vector<int>> blocks_by_definition(int n, const PlainRun &run) {
  const uint32_t low = 7u;
  const int no = (int)run.ops.size(), most_high = std::min(4, n - 3);
  std::vector<char> done(no, 0);
  std::vector<std::vector<int>> out;
  for (int left = no; left;) {
    std::vector<int> best;
    int most = 0;
    for (int force = -1; force < n; ++force) {
      if (force >= 0 && force < 3) continue;
      uint32_t T = force < 0 ? 0 : 1u << force, blocked = 0;
      std::vector<int> cur;
      int ops = 0;
      for (int i = 0; i < no; ++i) {
        if (done[i]) continue;
        const TileOp &op = run.ops[i];
        const uint32_t m = (1u << op.d[0]) | (op.kind == TOP_CX ? 1u << op.d[1] : 0u), t2 = T | (m & ~low);
        if ((m & blocked) || __builtin_popcount(t2) > most_high) {
          blocked |= m;
        } else {
          T = t2;
          cur.push_back(i);
          ops += run.count[i];
        }
      }
      if (ops > most) {
        most = ops;
        best = cur;
      }
    }
    for (int i : best) done[i] = 1;
    left -= (int)best.size();
    out.push_back(best);
  }
  return out;
}

static int blocks() {
  int bad = 0;
  for (int trial = 0; trial < 1000; ++trial) {
    const int n = uni(7, 18), nops = uni(1, 100), lo = uni(0, 2), hi = n - 1 - uni(0, 2);
    PlainRun run;
    std::vector<double> prm(kMap, kMap + 12);
    prm.insert(prm.end(), kScale, kScale + 16);
    const double noise[3] = {0.99, 0.8, 0.97};
    prm.insert(prm.end(), noise, noise + 3);
    int total = 0;
    for (int i = 0; i < nops; ++i) {
      dm_op op;
      memset(&op, 0, sizeof(op));
      const int r = uni(0, 19);
      op.kind = r < 11 ? DM_OP_1Q : r < 15 ? DM_OP_CX : r < 19 ? DM_OP_CX_SCALED : DM_OP_MEMORY_NOISE;
      op.param = r < 11 ? 0 : r < 19 ? 12 : 28;
      op.qubits[0] = uni(lo, hi);
      do op.qubits[1] = uni(lo, hi);
      while (op.qubits[1] == op.qubits[0]);
      add_plain(n, op, prm.data(), i, &run);
      total += op.kind == DM_OP_MEMORY_NOISE ? n : 1;
    }
    settle_all(n, &run);
    int counted = 0;
    for (int c : run.count) counted += c;
    if (counted != total || run.total != total) ++bad;
    if (plain_blocks(n, run) != blocks_by_definition(n, run)) ++bad;
  }
  return bad;
}

int main() {
  const int a = stages(), b = blocks();
  printf("stages %d blocks %d\n", a, b);
  return a || b;
}
'''

LONG = COMMON + r'''
// gates on digits lo..hi, the last gate on `late` if it is >= 0
static void long_program(int gates, int lo, int hi, int late, std::vector<TileOp> *ops, std::vector<double> *vals) {
  for (int i = 0; i < gates; ++i) {
    TileOp op;
    memset(&op, 0, sizeof(op));
    op.param = (int32_t)vals->size();
    op.d[0] = uni(lo, hi);
    op.kind = uni(0, 9) < 6 ? TOP_1Q : TOP_CX;
    do op.d[1] = uni(lo, hi);
    while (op.d[1] == op.d[0]);
    op.k = op.kind == TOP_CX;
    if (late >= 0 && i == gates - 1) {
      op.kind = TOP_1Q;
      op.d[0] = late;
    }
    const double *v = op.kind == TOP_1Q ? kMap : kScale;
    vals->insert(vals->end(), v, v + (op.kind == TOP_1Q ? 12 : 16));
    ops->push_back(op);
  }
}

int main() {
  const int gates = 400000;
  for (int m = 6; m <= 7; ++m)
    for (int late = 0; late < 2; ++late)
      for (int ordered = 0; ordered < 2; ++ordered) {
        std::vector<TileOp> ops;
        std::vector<double> vals;
        long_program(gates, 0, m - 2, late ? m - 1 : -1, &ops, &vals);
        const auto t0 = std::chrono::steady_clock::now();
        RegPlan rp;
        if (ordered) reg_plan(reg_items_in_order(ops, vals), m, false, true, &rp);
        else reg_plan(reg_items(ops, vals, m), m, false, false, &rp);
        printf("digits %d late %d ordered %d: %.2f s, %d stages\n", m, late, ordered,
               std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count(), rp.ns);
        fflush(stdout);
      }
  for (int n = 8; n <= 16; n += 8)
    for (int late = 0; late < 2; ++late) {
      std::vector<TileOp> ops;
      std::vector<double> vals;
      long_program(gates, 1, n - 1, late ? 0 : -1, &ops, &vals);
      const auto t0 = std::chrono::steady_clock::now();
      PlainRun run;
      for (size_t i = 0; i < ops.size(); ++i)
        push_plain(ops[i], vals.data() + ops[i].param, ops[i].kind == TOP_1Q ? 12 : 16, (int)i, &run);
      printf("positions %d late %d: %zu blocks", n, late, plain_blocks(n, run).size());
      printf(", %.2f s\n", std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
      fflush(stdout);
    }
  return 0;
}
'''


CHOICE = COMMON + r'''
// Whether a run of `gates` single-qubit and CX gates on the qubits 0-3, each
// followed by a memory-noise level if noise is not null, becomes passes.
static bool fuses(int n, int gates, const double *noise) {
  std::vector<double> prm(kMap, kMap + 12);
  if (noise) prm.insert(prm.end(), noise, noise + 3);
  PlainRun run;
  uint32_t used = 0;
  for (int i = 0; i < gates; ++i)
    for (int level = 0; level < (noise ? 2 : 1); ++level) {
      dm_op op;
      memset(&op, 0, sizeof(op));
      op.kind = level ? DM_OP_MEMORY_NOISE : i % 8 < 4 ? DM_OP_1Q : DM_OP_CX;
      op.param = level ? 12 : 0;
      op.qubits[0] = i % 4;
      op.qubits[1] = (i + 1) % 4;
      add_plain(n, op, prm.data(), i, &run);
      used |= plain_positions(n, op);
    }
  settle_all(n, &run);
  const size_t blocks = n <= 6 ? 1 : plain_blocks(n, run).size();
  if (least_blocks(used) > blocks) abort();
  return plain_pass_cost(n, blocks) < run.kernels;
}

int main() {
  const double dephasing[3] = {0.998, 1.0, 1.0}, thermal[3] = {0.998, 1.0, 0.999};
  struct {
    int n, gates;
    const double *noise;
    double kernels, passes;  // us a call, measured
  } rows[] = {{5, 4, thermal, 63, 33},   {5, 8, nullptr, 41, 33},   {7, 4, nullptr, 24, 32}, {7, 2, dephasing, 23, 32},
              {7, 1, thermal, 26, 33},   {7, 2, thermal, 39, 33},   {9, 4, nullptr, 27, 34}, {9, 8, nullptr, 43, 35},
              {9, 4, dephasing, 42, 46}, {9, 8, dephasing, 64, 48}, {10, 4, nullptr, 39, 35}, {11, 4, nullptr, 65, 38},
              {12, 2, nullptr, 104, 58}, {13, 4, thermal, 3800, 606}};
  int bad = 0;
  for (const auto &r : rows)
    if (fuses(r.n, r.gates, r.noise) != (r.passes < r.kernels)) {
      printf("%d qubits, %d gates: the slower choice\n", r.n, r.gates);
      ++bad;
    }
  return bad;
}
'''


COMPOSE = COMMON + r'''
// Composed maps are rounded once: every value of a run of single-qubit maps
// and noise levels on one position, and of the item made of it, against the
// product in 113 bits.
typedef __float128 Q;

int main() {
  int bad = 0;
  double worst = 0.0;
  for (int trial = 0; trial < 300; ++trial) {
    const int n = 7, q = 3, nops = uni(2, 120);
    Q e[12] = {0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
    PlainRun run;
    std::vector<TileOp> ops;
    std::vector<double> vals;
    for (int i = 0; i < nops; ++i) {
      double R[12] = {0};
      dm_op op;
      memset(&op, 0, sizeof(op));
      std::vector<double> prm;
      if (uni(0, 2)) {
        op.kind = DM_OP_MEMORY_NOISE;
        const double g = 0.9 + 0.099 * uni(0, 1000) / 1000.0, f = 0.9 + 0.0001 * uni(0, 1000), p = 0.001 * uni(0, 1000);
        prm = {f, p, g};
        R[1] = R[6] = sqrt(g) * f;
        R[8] = (1 - g) * (2 * p - 1);
        R[11] = g;
      } else {
        op.kind = DM_OP_1Q;
        op.qubits[0] = q;
        const double a = 0.01 * uni(0, 628), b = 0.01 * uni(0, 628), ca = cos(a), sa = sin(a), cb = cos(b), sb = sin(b);
        const double U[9] = {ca, -sa * cb, sa * sb, sa, ca * cb, -ca * sb, 0, sb, cb};
        for (int r = 0; r < 3; ++r)
          for (int c = 0; c < 3; ++c) R[4 * r + 1 + c] = U[3 * r + c];
        prm.assign(R, R + 12);
      }
      add_plain(n, op, prm.data(), i, &run);
      TileOp t;
      memset(&t, 0, sizeof(t));
      t.kind = TOP_1Q;
      t.k = 1;
      t.param = (int32_t)vals.size();
      ops.push_back(t);
      vals.insert(vals.end(), R, R + 12);
      Q w[12];
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 4; ++c) {
          w[4 * r + c] = c ? Q(0) : Q(R[4 * r]);
          for (int k = 0; k < 3; ++k) w[4 * r + c] += Q(R[4 * r + 1 + k]) * e[4 * k + c];
        }
      for (int c = 0; c < 12; ++c) e[c] = w[c];
    }
    settle_all(n, &run);
    int at = -1;
    for (size_t i = 0; i < run.ops.size(); ++i)
      if (run.ops[i].d[0] == n - 1 - q) at = run.ops[i].param;
    const std::vector<RegItem<long double>> items = reg_items(ops, vals, 7);
    if (items.size() != 1) ++bad;
    for (int c = 0; c < 12 && at >= 0; ++c) {
      const double v[2] = {(double)run.vals[at + c], (double)items[0].v[c]};
      // half a unit in the last place, and the 64-bit roundings of the chain
      const double tol = ldexp(fabs((double)e[c]), -53) + ldexp(4.0 * nops, -64);
      for (double x : v) {
        const double err = fabs((double)(Q(x) - e[c]));
        worst = std::max(worst, err / tol);
        if (!(err <= tol)) ++bad;
      }
    }
    if (at < 0) ++bad;
  }
  printf("%d above, worst %.2f of the bound\n", bad, worst);
  return bad != 0;
}
'''


def run_driver(tmp_path, source, limit):
    if shutil.which('g++') is None:
        pytest.skip('no g++')
    drv, exe = tmp_path / 'driver.cpp', tmp_path / 'driver'
    drv.write_text(source)
    subprocess.run(['g++', '-std=c++17', '-O2', '-Wall', '-Werror', '-Wno-unused-function', '-Wno-unused-variable',
                    '-I', os.path.join(ROOT, 'include'), '-I', os.path.join(ROOT, 'qiskit-aakash_amd', 'csrc'),
                    str(drv), '-o', str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=limit)
    assert res.returncode == 0, res.stdout + res.stderr
    return res.stdout


def test_stages_and_blocks_follow_their_definition(tmp_path):
    assert run_driver(tmp_path, DEFINITION, 60).strip() == 'stages 0 blocks 0'


def test_planning_time_goes_with_the_program(tmp_path):
    assert len(run_driver(tmp_path, LONG, 20).splitlines()) == 12


def test_runs_are_fused_where_that_was_measured_faster(tmp_path):
    run_driver(tmp_path, CHOICE, 20)


def test_composed_maps_are_rounded_once(tmp_path):
    run_driver(tmp_path, COMPOSE, 20)
