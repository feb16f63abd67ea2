"""Benchmark: noisy gates/s of the density-matrix update path on one MI355X.

Workload (the headline case): 16 qubits (4^16 Pauli coefficients), 1000
seeded gates -- U3 with probability 0.6 (angles U[0, 2pi)), else CX on
(q, q +- d), d ~ Geometric(0.5) -- each followed by a depolarising channel
p = 1e-3 on its qubits.  One step applies the whole 1000-gate program to the
resident state.

Paths measured:
  plain_fp64   one kernel per noisy gate, FP64 storage (the baseline);
  fused_fp32   gates fused into tile passes (one HBM round trip per block of
               gates, applied in LDS), FP32 storage, partition chosen by the
               learned cost model when a trained model is available, else by
               the greedy rule (the chosen method is reported in
               config.fusion).
``value`` is the fused FP32 throughput; the plain FP64 figure, the speed-up
and the accuracy of the FP32 result against FP64 are reported beside it.

Timing: the fused FP32 program runs once (accuracy against FP64), then
``warmup`` + ``steps`` times; the plain FP64 program, ~11 s per application,
is timed on ``--plain-steps`` (default 1) applications, so the driver's
``--steps 20 --warmup 5`` finishes in about a minute of GPU time.  The JSON
line is printed before any optional work (``--all-paths``).

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--plain-steps P] [--no-cpu-baseline]
                       [--all-paths]
       python bench.py --config precision|thermal|batch
       python bench.py --kernels | --kernels-dense | --tile-ops   (short runs for rocprofv3)
"""
import argparse
import json
import math
import os
import re
import sys
import time

os.environ.setdefault('OMP_NUM_THREADS', '1')  # the CPU baseline is a one-core numpy run
ROOT = os.path.dirname(os.path.abspath(__file__))
for _p in (ROOT, os.path.join(ROOT, 'qiskit-aakash_amd')):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import numpy as np  # noqa: E402

from dmsim import fusion, native, ptm, workloads  # noqa: E402

HBM_PEAK_GBS = 8000.0
# HBM bytes per launch measured with rocprofv3 FETCH_SIZE / WRITE_SIZE passes
# over `bench.py --kernels`, each divided by the counter's reading on a pass
# of known traffic (the diagonal memory-noise pass)
TRAFFIC_FILE = os.path.join(ROOT, 'profiles', 'headline_16q_hbm_traffic.md')
MFMA_PEAK_TFLOPS = {'fp32': 157.3, 'fp64': 78.6}
METRIC = 'noisy gates/sec at 16q: learned-fused FP32 vs plain FP64; % HBM peak'


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def zero_state(st, n):
    st.init_product(np.tile([1.0, 0.0, 0.0, 1.0], n), 0.5 ** n)


class PlainProgram:
    """One kernel per noisy gate: a program of its own for every gate (the
    library fuses the single operations of one FP64 program)."""

    def __init__(self, noisy, n):
        self.programs = [fusion.plain_program([g], n) for g in noisy]

    def __len__(self):
        return len(self.programs)

    def run(self, st):
        for prog in self.programs:
            prog.run(st)


def time_program(prog, n, precision, steps, warmup, st=None):
    """Wall time of `steps` program applications (after `warmup`), with HIP
    event timing of every launch on the handle's stream.  With ``st`` given
    the applications continue on that state (left open); otherwise a fresh
    |0..0> state is made and closed."""
    own = st is None
    if own:
        st = native.DeviceState(n, precision)
        zero_state(st, n)
    for _ in range(warmup):
        prog.run(st)
    st.synchronize()
    st.profile(True)
    st.profile_reset()
    t0 = time.perf_counter()
    for _ in range(steps):
        prog.run(st)
    st.synchronize()
    t1 = time.perf_counter()
    fams = {f: st.profile_read(f) for f in native.FAMILIES}
    st.profile(False)
    if own:
        st.close()
    return t1 - t0, fams


def kernel_roofline(fams, n, precision):
    """Roofline of the kernel family with the largest total time."""
    s = 8 if precision == 'fp64' else 4
    N = 4 ** n
    dom = max(fams, key=lambda f: fams[f][1])
    launches, ms = fams[dom]
    avg_s = ms / 1e3 / max(1, launches)
    if dom == 'fused':
        # a tile pass reads and writes every coefficient once
        byts = 2.0 * N * s
        ach = byts / avg_s / 1e9
        return dom, {'bound': 'hbm', 'achieved': ach, 'peak': HBM_PEAK_GBS, 'unit': 'GB/s',
                     'frac': ach / HBM_PEAK_GBS, 'traffic': None}, avg_s, byts, 0.0
    if dom in ('block3', 'block4'):
        k = 3 if dom == 'block3' else 4
        flops = 2.0 * 4 ** k * N
        byts = 2.0 * N * s
        intensity = flops / byts
        ridge = MFMA_PEAK_TFLOPS[precision] * 1e12 / (HBM_PEAK_GBS * 1e9)
        if intensity >= ridge:
            return dom, {'bound': 'mfma', 'achieved': flops / avg_s / 1e12, 'peak': MFMA_PEAK_TFLOPS[precision],
                         'unit': 'TFLOP/s', 'frac': flops / avg_s / 1e12 / MFMA_PEAK_TFLOPS[precision],
                         'traffic': None}, avg_s, byts, flops
        ach = byts / avg_s / 1e9
        return dom, {'bound': 'hbm', 'achieved': ach, 'peak': HBM_PEAK_GBS, 'unit': 'GB/s',
                     'frac': ach / HBM_PEAK_GBS, 'traffic': None}, avg_s, byts, flops
    per = {'1q': 2 * 0.75, 'cx': 2 * 15 / 16, '2q': 2 * 15 / 16, 'memory_noise': 2.0, 'diag': 2.0}.get(dom, 2.0)
    byts = per * N * s
    ach = byts / avg_s / 1e9
    return dom, {'bound': 'hbm', 'achieved': ach, 'peak': HBM_PEAK_GBS, 'unit': 'GB/s',
                 'frac': ach / HBM_PEAK_GBS, 'traffic': None}, avg_s, byts, 0.0


def measured_traffic(key, plan):
    """Recorded HBM bytes per launch of kernel family ``key`` under ``plan``
    ('learned/104', or 'any' for plan-independent kernels), or None."""
    try:
        with open(TRAFFIC_FILE) as f:
            text = f.read()
    except OSError:
        return None
    m = re.search(r'^traffic_bytes_per_launch %s %s: ([0-9.eE+]+)\s*$' % (re.escape(key), re.escape(plan)), text,
                  re.M)
    return float(m.group(1)) if m else None


def streaming_fraction(fams, n, precision, counts):
    """Sum of compulsory bytes of the plain streaming kernels / their time / peak."""
    s = 8 if precision == 'fp64' else 4
    N = 4 ** n
    tot_b = tot_t = 0.0
    for fam, per in (('1q', 1.5), ('cx', 2 * 15 / 16), ('2q', 2 * 15 / 16)):
        launches, ms = fams[fam]
        if launches:
            tot_b += per * N * s * launches
            tot_t += ms / 1e3
    return (tot_b / tot_t / 1e9 / HBM_PEAK_GBS) if tot_t else None


def accuracy(st32, st64, n):
    """FP32 state against the FP64 state of the same program applied to
    |0..0>, compared on the device in FP64: max coefficient error, fidelity
    (normalised overlap), trace and purity, and the n single-qubit marginals
    P(q = 0)."""
    cmp = st32.compare(st64)
    tr, pur = st32.trace_purity()
    m32 = np.array([st32.probabilities([q], 'Z')[0] for q in range(n)])
    m64 = np.array([st64.probabilities([q], 'Z')[0] for q in range(n)])
    a0 = float(st32.read([0])[0])
    return {'max_abs_coeff_err': cmp['max_abs_diff'], 'max_abs_coeff_err_x2n': cmp['max_abs_diff'] * 2.0 ** n,
            'fidelity_fp32_vs_fp64': cmp['dot'] / cmp['norm2_other'], 'trace_fp32': tr, 'purity_fp32': pur,
            'purity_fp64': cmp['norm2_other'] * 2.0 ** n, 'max_marginal_err': float(np.max(np.abs(m32 - m64))),
            'identity_coeff_exact': a0 == 2.0 ** -n}


def host_cpu():
    """(logical CPUs, CPU model) of this host."""
    model = None
    try:
        with open('/proc/cpuinfo') as f:
            for line in f:
                if line.startswith('model name'):
                    model = line.split(':', 1)[1].strip()
                    break
    except OSError:
        pass
    return os.cpu_count(), model


def cpu_baseline(n_target, G, seed, budget_s=20.0, n_sample=13):
    """The oracle (FP64 numpy restatement of the reference, one core) on the
    same workload generator at `n_sample` qubits until `budget_s` elapses;
    gates/s scaled to `n_target` qubits by 4^-(n_target - n_sample) (the work
    per gate is proportional to 4^n)."""
    from oracle import refsim
    n = n_sample
    gates = workloads.local_u3_cx(n, G, seed)
    st = refsim.initial_state(n)
    done = 0
    t0 = time.perf_counter()
    for name, qs, prm in gates:
        if name == 'u3':
            q = qs[0]
            s3 = st.reshape(4 ** q, 4, 4 ** (n - q - 1))
            for axis, ang in refsim.gate_rotations('u3', prm):
                s3 = refsim.rotate_components(s3, axis, ang, [1.0, 0.0])
            st = refsim.apply_gate_depolarizing(s3.reshape(n * [4]), n, [q], 1e-3)
        else:
            st = refsim.apply_cx(st, qs[0], qs[1], [1.0, 0.0], n)
            st = refsim.apply_gate_depolarizing(st, n, list(qs), 1e-3)
        done += 1
        if time.perf_counter() - t0 > budget_s:
            break
    el = time.perf_counter() - t0
    rate = done / el
    ncpu, model = host_cpu()
    return {'value': rate / 4 ** (n_target - n), 'unit': 'gates/s', 'cores': 1, 'kind': 'port',
            'host_logical_cpus': ncpu, 'cpu_model': model,
            'sample': '%d gates of the same generator at %d qubits (FP64 oracle, numpy, 1 thread) in %.1f s = '
                      '%.3f gates/s; scaled by 4^-%d to %d qubits' % (done, n, el, rate, n_target - n, n_target)}


def headline_plan(noisy, n, fusion_arg='auto', precision='fp32'):
    """(program, blocks, method, plan seconds) of the headline fused path:
    the learned planner when the trained model ships, else greedy; tiles
    and costs for a state of the given precision."""
    method = fusion_arg
    cost = None
    if method in ('auto', 'learned'):
        try:
            from dmsim import costmodel
            cost = costmodel.default_model()
            cost.precision = precision
            method = 'learned'
        except Exception as e:  # no trained model shipped
            if fusion_arg == 'learned':
                raise
            log('no learned cost model (%s); greedy fusion' % e)
            method = 'greedy'
    t0 = time.perf_counter()
    prog, blocks = fusion.fused_program(noisy, n, fusion.KMAX[method], method, cost, 'seq', precision=precision)
    return prog, blocks, method, time.perf_counter() - t0


def kernels_mode(args):
    """One short run for rocprofv3 counter passes, in this order:
      1. calibration: a diagonal memory-noise pass (k_diag_pow), which reads
         and writes every coefficient exactly once (N*s bytes each way), FP64
         then FP32, 3 launches each;
      2. one application of the headline fused FP32 program (same plan);
      3. the first 60 gates of the plain FP64 program."""
    from dmsim.program import Program
    n, G = args.qubits, args.gates
    noisy = fusion.noisy_gates(workloads.local_u3_cx(n, G, args.seed), 1e-3)
    fused, blocks, method, _ = headline_plan(noisy, n, args.fusion)
    out = {'n': n, 'plan': '%s/%d' % (method, len(fused)), 'calib_launches': 3}
    for prec in ('fp64', 'fp32'):
        st = native.DeviceState(n, prec)
        zero_state(st, n)
        prog = Program(n)
        for _ in range(3):
            prog.memory_noise(0.99, 0.5, 0.98)   # thermal feed (1-g)(2p-1) = 0: one diagonal pass
        prog.run(st)
        st.synchronize()
        if prec == 'fp32':
            fused.run(st)
            st.synchronize()
        st.close()
    st = native.DeviceState(n, 'fp64')
    zero_state(st, n)
    PlainProgram(noisy[:60], n).run(st)
    st.synchronize()
    st.close()
    return out


def dense_kernels_mode(args):
    """One short run of the matrix-core kernels at n qubits (for rocprofv3
    MFMA counter passes): per precision, the standalone block kernel
    (dm_apply_block) and the dense tile pass, each for a 3- and a 4-qubit
    block PTM, 2 launches each, in this order."""
    from dmsim.program import Program
    n = args.qubits
    rng = np.random.default_rng(args.seed)
    out = {'n': n, 'order': []}
    for prec in ('fp32', 'fp64'):
        st = native.DeviceState(n, prec)
        zero_state(st, n)
        for k in (3, 4):
            qs = list(range(k))
            S = np.eye(4 ** k)
            S[1:, 1:] = rng.normal(size=(4 ** k - 1, 4 ** k - 1)) / 4 ** k
            for form in ('block', 'tile'):
                prog = Program(n)
                for _ in range(2):
                    if form == 'block':
                        prog.block(qs, S)
                    else:
                        prog.fused(6, qs, [(native.SUB_DENSE, qs, S)])
                prog.run(st)
                st.synchronize()
                out['order'].append('%s_%s_k%d' % (prec, form, k))
        st.close()
    return out


def tile_ops_mode(args):
    """Per-operation cost of tile passes at n qubits, FP32 (also a short run
    for rocprofv3 LDS counter passes): for 6- and 7-digit tiles over the
    highest qubits, one launch each of a pass with no operations, then with 8
    copies of one operation: a 1q PTM on a high digit, on tile digit 0 and on
    tile digit 1, a CX on two high digits, on digits 0 and 1, on digit 2 and
    the highest digit, on digits 1 and 3 and on digits 2 and 4 (swizzled
    where they touch digits 0-2).
    Returns the milliseconds of each pass (HIP events)."""
    from dmsim.program import Program
    n = args.qubits
    R = ptm.rows3(ptm.depolarizing1(1e-3) @ ptm.gate_ptm('u3', [0.3, 0.2, 0.1]))
    S = ptm.depolarizing_pair_scale(1e-3)
    lo = [n - 1, n - 2, n - 3]   # qubits at positions 0, 1, 2 (tile digits 0, 1, 2)
    st = native.DeviceState(n, 'fp32')
    zero_state(st, n)
    out = {'n': n, 'ms': {}}
    for m, qs in ((6, [0, 1, 2]), (7, [0, 1, 2, 3])):
        hi = qs[::-1]   # tile digits 3, 4, ...
        cases = [('empty', []), ('1q high', [(native.SUB_1Q, [0], R)]), ('1q d0', [(native.SUB_1Q, [lo[0]], R)]),
                 ('1q d1', [(native.SUB_1Q, [lo[1]], R)]), ('cx high', [(native.SUB_CX, [0, 1], S)]),
                 ('cx d0 d1', [(native.SUB_CX, [lo[0], lo[1]], S)]), ('cx d2 high', [(native.SUB_CX, [lo[2], 0], S)]),
                 ('cx d1 d3', [(native.SUB_CX, [lo[1], hi[0]], S)]), ('cx d2 d4', [(native.SUB_CX, [lo[2], hi[1]], S)])]
        for label, sub in cases:
            prog = Program(n)
            prog.fused(m, qs, sub * 8)
            prog.run(st)   # upload and warm-up
            st.synchronize()
            st.profile(True)
            st.profile_reset()
            prog.run(st)
            st.synchronize()
            out['ms']['m%d %s' % (m, label)] = round(sum(st.profile_read(f)[1] for f in native.FAMILIES), 3)
            st.profile(False)
    st.close()
    return out


def parse_batch_choice(text):
    """'fp64=6/256/256,fp32=5/256/64' -> {precision: (lds_max_qubits,
    lds_threads, items_per_pass)}; '' -> {}."""
    out = {}
    for part in filter(None, (text or '').split(',')):
        prec, _, val = part.partition('=')
        if prec not in ('fp64', 'fp32'):
            raise ValueError('--batch-choice: unknown precision %r' % prec)
        vals = tuple(int(x) for x in val.split('/'))
        if len(vals) != 3:
            raise ValueError('--batch-choice: want lds_max_qubits/lds_threads/items_per_pass, got %r' % val)
        out[prec] = vals
    return out


def batch_mode(args):
    """Batched circuits (U3/CX 70/30, memory noise after every gate, Z
    ensemble at the end), FP64 and FP32, autotuned (or the --batch-choice
    given for a precision), hipGraph replay."""
    from dmsim import batch
    lo, hi = (int(x) for x in args.batch_widths.split('-'))
    count = args.batch_circuits
    specs = workloads.batch(count, args.seed, n_range=(lo, hi))
    fixed = parse_batch_choice(args.batch_choice)
    lines = {}
    programs = {}
    for prec in ('fp64', 'fp32'):
        if prec in fixed:
            (lmax, thr, ipp), tune = fixed[prec], {}
            log('%s: lds_max_qubits %d, %d threads, %d items per pass (given)' % (prec, lmax, thr, ipp))
        else:
            log('%s: autotuning ...' % prec)
            t0 = time.perf_counter()
            (lmax, thr, ipp), tune = batch.autotune(specs, prec, programs=programs)
            log('  chose lds_max_qubits %d, %d threads, %d items per pass (%.1f s)' % (lmax, thr, ipp,
                                                                                     time.perf_counter() - t0))
        t0 = time.perf_counter()
        batch.workload_programs(specs, prec, lmax)
        host_build_s = time.perf_counter() - t0
        b = batch.from_workload(specs, prec, lds_max_qubits=lmax, lds_threads=thr, items_per_pass=ipp,
                                programs=programs)
        info = b.info()
        for _ in range(args.warmup):
            b.run(True)
        t0 = time.perf_counter()
        us_all = []
        for _ in range(args.steps):
            _, us, ms = b.run(True)
            us_all.append(us)
        wall = time.perf_counter() - t0
        b.close()
        us = np.concatenate(us_all)
        lines[prec] = {'circuits_per_s': count * args.steps / wall, 'p50_us': float(np.percentile(us, 50)),
                       'p99_us': float(np.percentile(us, 99)), 'lds_max_qubits': lmax, 'lds_threads': thr,
                       'items_per_pass': ipp, 'hbm_tier': info, 'autotune_ms': tune.get('trials_ms'),
                       'host_build_s': host_build_s}
        log('%s: %s' % (prec, json.dumps(lines[prec])))
    return {'metric': 'circuits/sec, %d noisy circuits of %d-%d qubits (one hipGraph: LDS-tier launches + one '
                      'launch per round of HBM-tier passes)' % (count, lo, hi),
            'value': lines['fp64']['circuits_per_s'], 'unit': 'circuits/s', 'n_gpus': 1, 'steps': args.steps,
            'warmup': args.warmup, 'higher_is_better': True, 'dtype': 'f64', 'data': 'synthetic',
            'config': {'workload': '%d circuits, widths U{%d..%d}, gates U{50..300} (U3 0.7 / CX 0.3), decay and '
                                   'depolarisation rates logU[1e-4,1e-2], barrier after every gate, seed %d'
                                   % (count, lo, hi, args.seed), 'fp64': lines['fp64'], 'fp32': lines['fp32']}}


def precision_mode(args):
    """17 qubits, FP32 and FP64 states resident together, each running the
    fused program planned for its precision, as the backend plans it
    (depolarising 5e-4 per gate); errors on the device."""
    n = 17
    gates = workloads.matching_layers(n, args.layers, args.seed)
    noisy = fusion.noisy_gates(gates, 5e-4)
    res = {}
    states = {}
    for prec in ('fp64', 'fp32'):
        prog, blocks, method, _ = headline_plan(noisy, n, args.fusion, prec)
        res['fusion'] = method
        res['passes_' + prec] = len(prog)
        log('precision config, %s: %d gates, %d passes (%s)' % (prec, len(noisy), len(prog), method))
        st = native.DeviceState(n, prec)
        zero_state(st, n)
        st.synchronize()
        t0 = time.perf_counter()
        prog.run(st)
        st.synchronize()
        res[prec + '_gates_per_s'] = len(noisy) / (time.perf_counter() - t0)
        log('  %s: %.1f gates/s' % (prec, res[prec + '_gates_per_s']))
        states[prec] = st
    cmp = states['fp32'].compare(states['fp64'])
    fid = cmp['dot'] / math.sqrt(cmp['norm2_self'] * cmp['norm2_other'])
    m32 = [states['fp32'].probabilities([q], 'Z')[0] for q in range(n)]
    m64 = [states['fp64'].probabilities([q], 'Z')[0] for q in range(n)]
    for st in states.values():
        st.close()
    res.update({'max_abs_coeff_err': cmp['max_abs_diff'], 'max_abs_coeff_err_x2n': cmp['max_abs_diff'] * 2.0 ** n,
                'fidelity_overlap': fid, 'purity_fp64': cmp['norm2_other'] * 2.0 ** n,
                'purity_fp32': cmp['norm2_self'] * 2.0 ** n,
                'max_marginal_err': float(np.max(np.abs(np.array(m32) - np.array(m64)))),
                'marginals_fp64': m64, 'gates': len(noisy)})
    log(json.dumps(res))
    return {'metric': '17-qubit FP32 vs FP64 accuracy and throughput (fused)', 'value': res['fp32_gates_per_s'],
            'unit': 'gates/s', 'n_gpus': 1, 'higher_is_better': True, 'dtype': 'f32', 'data': 'synthetic',
            'config': dict(res, workload='17q, %d layers of U3 on every qubit + CX on a random perfect matching, '
                                          'depolarising 5e-4 per gate, seed %d' % (args.layers, args.seed))}


def thermal_mode(args):
    """14 qubits, 30 brickwork layers + QFT, thermal relaxation (T1 = 50 us,
    T2 = 70 us, 50 ns gates) after every gate, partial Z measure of qubits 0-3,
    through the backend (execute) in FP64."""
    from dmsim import BasicAer, execute
    n = 14
    g, f = workloads.thermal_factors(50e-6, 70e-6, 50e-9)
    gates = workloads.brickwork_qft(n, 30, args.seed)
    qc = workloads.to_circuit(n, gates, barrier_after_each=True, measure=('partial', [0, 1, 2, 3], 'Z'))
    be = BasicAer.get_backend('dm_simulator')
    out = {}
    for fusion_mode in ('none', 'greedy', 'learned'):
        t0 = time.perf_counter()
        r = execute(qc, be, decay_factor=g, decoherence_factor=f, thermal_factor=1.0,
                    compute_densitymatrix=False, fusion=fusion_mode).result()
        wall = time.perf_counter() - t0
        res = r['results'][0]
        out[fusion_mode] = {'wall_s': wall, 'running_time_taken': res['running_time_taken'],
                            'levels': res['number_of_clock_cycles'],
                            'partial_probability': res['data']['partial_probability'],
                            'trace': float(res['data']['coeffmatrix'][0] * 2 ** n)}
        log('%s: %s' % (fusion_mode, json.dumps({k: v for k, v in out[fusion_mode].items()
                                                  if k != 'partial_probability'})))
    pp = out['none']['partial_probability']
    return {'metric': '14-qubit thermal brickwork+QFT, gates/s (FP64, execute)',
            'value': len(gates) / out['none']['running_time_taken'], 'unit': 'gates/s', 'n_gpus': 1,
            'higher_is_better': True, 'dtype': 'f64', 'data': 'synthetic',
            'config': {'workload': '14q, 30 brickwork layers + QFT, T1=50us T2=70us dt=50ns, barrier after every '
                                   'gate, partial Z on q0-3', 'plain': out['none'], 'fused': out['greedy'],
                       'fused_learned': out['learned'],
                       'fused_gates_per_s': len(gates) / out['greedy']['running_time_taken'],
                       'fused_learned_gates_per_s': len(gates) / out['learned']['running_time_taken'],
                       'max_partial_prob_diff_fused_vs_plain': max(
                           abs(pp[k] - out[m]['partial_probability'][k]) for m in ('greedy', 'learned') for k in pp)}}


def parse_args(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument('--gpus', type=int, default=1)
    ap.add_argument('--steps', type=int, default=2)
    ap.add_argument('--warmup', type=int, default=1)
    ap.add_argument('--qubits', type=int, default=16)
    ap.add_argument('--gates', type=int, default=1000)
    ap.add_argument('--seed', type=int, default=0)
    ap.add_argument('--no-cpu-baseline', action='store_true')
    ap.add_argument('--no-accuracy', action='store_true')
    ap.add_argument('--fusion', default='auto', choices=['auto', 'greedy', 'search', 'learned'])
    ap.add_argument('--plain-steps', type=int, default=1, help='timed applications of the plain FP64 program')
    ap.add_argument('--all-paths', action='store_true',
                    help='after the headline line, also time plain FP32, fused FP64 and the greedy forms (stderr)')
    ap.add_argument('--config', default='headline', choices=['headline', 'batch', 'precision', 'thermal'])
    ap.add_argument('--layers', type=int, default=400, help='precision config: layers')
    ap.add_argument('--kernels', action='store_true', help='short per-kernel run (for rocprofv3 counters)')
    ap.add_argument('--kernels-dense', action='store_true', help='short matrix-core kernel run (MFMA counters)')
    ap.add_argument('--tile-ops', action='store_true', help='per-operation cost of tile passes (LDS counters)')
    ap.add_argument('--batch-circuits', type=int, default=512, help='batch config: circuits')
    ap.add_argument('--batch-widths', default='6-12', help='batch config: qubit range lo-hi')
    ap.add_argument('--batch-choice', default='',
                    help='batch config: fixed lds_max_qubits/lds_threads/items_per_pass per precision instead of '
                         'autotuning, e.g. fp64=6/256/256,fp32=5/256/64')
    return ap.parse_args(argv)


def main():
    args = parse_args()
    if args.gpus != 1:
        print('bench.py runs on one GPU: the path has no multi-GPU form in this build (--gpus %d refused)'
              % args.gpus, file=sys.stderr)
        sys.exit(2)

    if args.kernels:
        print(json.dumps(kernels_mode(args)), flush=True)
        return
    if args.kernels_dense:
        print(json.dumps(dense_kernels_mode(args)), flush=True)
        return
    if args.tile_ops:
        print(json.dumps(tile_ops_mode(args)), flush=True)
        return
    if args.config != 'headline':
        fn = {'batch': batch_mode, 'precision': precision_mode, 'thermal': thermal_mode}[args.config]
        print(json.dumps(fn(args)), flush=True)
        return

    headline(args)


def planned_applications(args):
    """Whole-program applications of the 1000-gate workload each path makes
    in a default headline run (the bound a CPU test checks): plain FP64 is
    timed on ``--plain-steps`` applications after one warm-up over its first
    PLAIN_WARMUP_GATES gates; the fused FP32 program runs once for the
    accuracy comparison, then ``warmup`` + ``steps`` times."""
    return {'plain_fp64': args.plain_steps + PLAIN_WARMUP_GATES / max(1, args.gates),
            'fused_fp32': 1 + args.warmup + args.steps,
            'other_paths': 6 * (1 + 2) if args.all_paths else 0}


# gates of the plain FP64 program run once before its timed applications
# (first launches of each kernel variant); one full application takes ~11 s
PLAIN_WARMUP_GATES = 100


def headline(args):
    n, G = args.qubits, args.gates
    gates = workloads.local_u3_cx(n, G, args.seed)
    noisy = fusion.noisy_gates(gates, 1e-3)

    fused, blocks, method, plan_s = headline_plan(noisy, n, args.fusion)
    plain = PlainProgram(noisy, n)
    ks = [len(q) if len(m) > 1 else 0 for q, m in blocks]
    log('plan: %s, %d passes for %d gates (%.2f s host); k histogram %s'
        % (method, len(fused), G, plan_s, np.bincount(ks, minlength=6).tolist()))

    # plain FP64: a short warm-up, then --plain-steps whole applications from
    # |0..0>; with one timed application the state is the FP64 reference the
    # FP32 result is compared with
    log('timing plain fp64 (%d application(s)) ...' % args.plain_steps)
    st64 = native.DeviceState(n, 'fp64')
    zero_state(st64, n)
    PlainProgram(noisy[:PLAIN_WARMUP_GATES], n).run(st64)
    zero_state(st64, n)
    t_plain, f_plain = time_program(plain, n, 'fp64', args.plain_steps, 0, st=st64)
    log('  %.3f s for %d application(s)' % (t_plain, args.plain_steps))
    if args.plain_steps != 1 and not args.no_accuracy:
        zero_state(st64, n)
        plain.run(st64)

    log('timing fused fp32 (%d warm-up, %d timed) ...' % (args.warmup, args.steps))
    st32 = native.DeviceState(n, 'fp32')
    zero_state(st32, n)
    fused.run(st32)
    acc = None
    if not args.no_accuracy:
        acc = accuracy(st32, st64, n)
        log('accuracy: %s' % json.dumps(acc))
    st64.close()
    t_fused, f_fused = time_program(fused, n, 'fp32', args.steps, args.warmup, st=st32)
    st32.close()
    log('  %.3f s for %d steps' % (t_fused, args.steps))

    dom, roof, avg_s, byts, flops = kernel_roofline(f_fused, n, 'fp32')
    pdom, proof, _, _, _ = kernel_roofline(f_plain, n, 'fp64')
    if n == 16 and G == 1000 and args.seed == 0:
        roof['traffic'] = measured_traffic('%s_fp32' % dom, '%s/%d' % (method, len(fused)))
        proof['traffic'] = measured_traffic('plain_fp64_%s' % pdom, 'any')
    cpu = None if args.no_cpu_baseline else cpu_baseline(n, G, args.seed)
    if cpu:
        log('cpu baseline: %s' % cpu['sample'])

    value = G * args.steps / t_fused
    plain_gps = G * args.plain_steps / t_plain
    step_s = t_fused / args.steps
    out = {
        'metric': METRIC,
        'value': value,
        'unit': 'gates/s',
        'n_gpus': 1,
        'steps': args.steps,
        'warmup': args.warmup,
        'ms_per_step': step_s * 1e3,
        'higher_is_better': True,
        'scaling': 'weak',
        'vs_baseline': None,
        'dtype': 'f32',
        'data': 'synthetic',
        'config': {
            'workload': '%dq local U3/CX 60/40 (CX distance ~ Geometric(0.5)), %d gates, depolarizing 1e-3 per '
                        'gate, seed %d' % (n, G, args.seed),
            'path': 'fused fp32 (%s partition, %d passes)' % (method, len(fused)),
            'fusion': method,
            'plain_fp64_gates_per_s': plain_gps,
            'plain_fp64_timed_applications': args.plain_steps,
            'speedup_fused_fp32_vs_plain_fp64': value / plain_gps,
            'plan_host_s': plan_s,
            'end_to_end_gates_per_s_incl_plan': G / (step_s + plan_s),
            'plain_fp64_dominant_kernel': pdom,
            'plain_fp64_roofline': proof,
            'plain_fp64_streaming_hbm_frac': streaming_fraction(f_plain, n, 'fp64', None),
            'fused_fp32_kernel_ms': {k: v[1] / max(1, v[0]) for k, v in f_fused.items() if v[0]},
            'fused_fp32_launches': {k: v[0] for k, v in f_fused.items() if v[0]},
            'accuracy_fp32_vs_fp64': acc,
        },
        'roofline': dict(roof, kernel=dom, avg_launch_ms=avg_s * 1e3, algorithmic_bytes=byts,
                         algorithmic_flops=flops),
        'cpu_baseline': cpu,
    }
    print(json.dumps(out), flush=True)

    if args.all_paths:
        # the other forms of the same workload, 1 warm-up + 2 timed steps each,
        # reported on stderr after the headline line
        extra = {}
        log('timing plain fp32, fused fp64 (FP32 plan and its own), greedy dense-MFMA fp32 ...')
        extra['plain_fp32'] = time_program(plain, n, 'fp32', 2, 1)
        extra['fused_fp64'] = time_program(fused, n, 'fp64', 2, 1)
        # the program an FP64 state gets from the planner (FP64 costs and tiles)
        fused64, _, _, _ = headline_plan(noisy, n, args.fusion, 'fp64')
        extra['fused_fp64_own_plan'] = time_program(fused64, n, 'fp64', 2, 1)
        dense, _ = fusion.fused_program(noisy, n, 4, 'greedy', None, 'dense')
        extra['greedy_dense_fp32'] = time_program(dense, n, 'fp32', 2, 1)
        dense3, _ = fusion.fused_program(noisy, n, 3, 'greedy', None, 'dense')
        extra['greedy_dense_k3_fp32'] = time_program(dense3, n, 'fp32', 2, 1)
        if method != 'greedy':
            gseq, _ = fusion.fused_program(noisy, n, 4, 'greedy', None, 'seq')
            extra['greedy_seq_fp32'] = time_program(gseq, n, 'fp32', 2, 1)
        log('other paths (gates/s): %s' % json.dumps({k: G * 2 / v[0] for k, v in extra.items()}))
        log('plain fp32 streaming HBM fraction: %s' % streaming_fraction(extra['plain_fp32'][1], n, 'fp32', None))


if __name__ == '__main__':
    main()
