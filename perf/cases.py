"""The workloads this engine's speed is judged on, each one call sequence of a
user's program through the public entry points.

Kinds of case:

* ``circuit``  -- a noisy circuit from |0..0> on a resident state: initialise,
  run the compiled program (``fusion.plain_program`` / ``fused_program`` and
  ``Program.run``), read the Z-ensemble probabilities.  The program and the
  state are kept by the caller, as a parameter sweep or a repeated run keeps
  them.  Outputs: all coefficients and the probabilities.
* ``execute``  -- the plugin interface, ``execute(circuit, backend, ...)``,
  from the circuit object to the result dictionary.
* ``batch``    -- many independent circuits in one submission
  (``batch.from_workload`` and ``Batch.run``).
* ``readout``  -- what is read from a finished state: ensemble and partial
  probabilities, trace and purity, the comparison with a second state, and
  on small registers the density matrix and the coefficients on the host.

The circuits are those of ``dmsim.workloads`` (uniform random U3/CX, local
U3/CX with geometric CX distances, layers over random matchings, brickwork),
with the noise the benchmark configurations use: per-gate depolarising, and
memory noise on every qubit (thermal relaxation or pure dephasing).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), 'qiskit-aakash_amd'))

from dmsim import BasicAer, batch, costmodel, execute, fusion, native, workloads  # noqa: E402

DEVICE = 'cuda' if torch.cuda.is_available() else 'cpu'

# T1 = 50 us, T2 = 70 us, 50 ns gates (the thermal configuration)
THERMAL = dict(zip(('decay', 'decoherence'), workloads.thermal_factors(50e-6, 70e-6, 50e-9)), thermal=1.0)
DEPHASING = {'decay': 1.0, 'decoherence': 0.998, 'thermal': 1.0}


def _circuit(name, n, gates, circuit, path, precision, depol=0.0, memory='none', every=0):
    return {'name': name, 'kind': 'circuit', 'n': n, 'gates': gates, 'circuit': circuit, 'path': path,
            'precision': precision, 'depol': depol, 'memory': memory, 'every': every}


def listed():
    return [
        # the smallest register a user runs gate by gate: launch latency
        _circuit('circuit_5q_fp64_plain', 5, 30, 'random', 'plain', 'fp64', memory='dephasing', every=5),
        # the CPU reference workload: 10 qubits, 200 random gates, one kernel per gate
        _circuit('circuit_10q_fp64_plain', 10, 200, 'random', 'plain', 'fp64', memory='thermal', every=10),
        # a notebook-sized run through the plugin interface, all outputs
        {'name': 'execute_8q_fp64', 'kind': 'execute', 'n': 8, 'gates': 40, 'circuit': 'random', 'fusion': 'none',
         'precision': 'fp64', 'memory': 'thermal'},
        # an odd width between cache-sized and large states, FP32
        _circuit('circuit_13q_fp32_learned', 13, 390, 'matching', 'learned', 'fp32', depol=5e-4),
        # thermal relaxation after every gate (the thermal configuration's circuit)
        _circuit('circuit_14q_fp64_greedy', 14, 100, 'brickwork', 'greedy', 'fp64', memory='thermal', every=1),
        # the backend's default precision with the learned planner, odd width
        _circuit('circuit_15q_fp64_learned', 15, 300, 'local', 'learned', 'fp64', depol=1e-3),
        # the headline benchmark: 16 qubits, 1000 local gates
        _circuit('circuit_16q_fp32_learned', 16, 1000, 'local', 'learned', 'fp32', depol=1e-3),
        # the plain baseline at full size: one kernel per noisy gate
        _circuit('circuit_16q_fp64_plain', 16, 40, 'local', 'plain', 'fp64', depol=1e-3),
        # the batching configuration in its tuned FP32 form
        {'name': 'batch_512_fp32_6to12', 'kind': 'batch', 'count': 512, 'nlo': 6, 'nhi': 12, 'dlo': 50, 'dhi': 300,
         'precision': 'fp32', 'lds_max': 6, 'threads': 1024},
        # many registers that fit one workgroup, FP64 (a parameter scan of small circuits)
        {'name': 'batch_512_fp64_2to7', 'kind': 'batch', 'count': 512, 'nlo': 2, 'nhi': 7, 'dlo': 50, 'dhi': 300,
         'precision': 'fp64', 'lds_max': 7, 'threads': 512},
        # everything read from a mid-size state, density matrix included
        {'name': 'readout_11q_fp64', 'kind': 'readout', 'n': 11, 'precision': 'fp64', 'other': 'fp64', 'measured': 4,
         'basis': 'X', 'dense': True},
        # large state: N-basis partial measurement, purity, FP32 against FP64
        {'name': 'readout_15q_fp32', 'kind': 'readout', 'n': 15, 'precision': 'fp32', 'other': 'fp64', 'measured': 7,
         'basis': 'N', 'dense': False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['circuit'] * 6 + ['batch'] * 2 + ['readout', 'execute'])
    precision = rng.choice(['fp64', 'fp32'])
    if kind == 'circuit':
        n = rng.randint(5, 16)
        path = rng.choice(['plain', 'greedy', 'learned', 'learned'])
        memory = rng.choice(['none', 'none', 'thermal', 'dephasing'])
        every = rng.choice([1, n, 3 * n]) if memory != 'none' else 0
        gates = _log_int(rng, 20, 1000)
        # at most about half a second at 5 TB/s: plain gates move the state
        # once each (noise up to four times), fused ones about a tenth of it
        per = 2.0 * 4 ** n * (8 if precision == 'fp64' else 4) / 5e12
        if path == 'plain':
            per *= 1.0 + (4.0 / every if every else 0.0)
        else:
            per *= 0.12 + (0.15 * n / every if every else 0.0)
        gates = max(10, min(gates, int(0.4 / per)))
        return {'kind': 'circuit', 'n': n, 'gates': gates,
                'circuit': rng.choice(['random', 'local', 'matching', 'brickwork']), 'path': path,
                'precision': precision, 'depol': rng.choice([0.0, 5e-4, 1e-3]), 'memory': memory, 'every': every}
    if kind == 'batch':
        nlo = rng.randint(2, 8)
        nhi = rng.randint(max(nlo, 5), 12)
        dlo = _log_int(rng, 10, 50)
        return {'kind': 'batch', 'count': _log_int(rng, 16, 512), 'nlo': nlo, 'nhi': nhi, 'dlo': dlo,
                'dhi': rng.randint(dlo + 10, 300), 'precision': precision, 'lds_max': rng.choice([5, 6, 7]),
                'threads': rng.choice([256, 512, 1024])}
    if kind == 'readout':
        n = rng.randint(6, 15)
        basis = rng.choice(['X', 'Y', 'Z', 'N'])
        return {'kind': 'readout', 'n': n, 'precision': precision, 'other': rng.choice(['fp64', 'fp32']),
                'measured': rng.randint(1, min(n, 8 if basis == 'N' else n)), 'basis': basis, 'dense': n <= 11}
    return {'kind': 'execute', 'n': rng.randint(3, 9), 'gates': rng.randint(20, 60),
            'circuit': rng.choice(['random', 'local']), 'fusion': rng.choice(['none', 'greedy', 'learned']),
            'precision': precision, 'memory': rng.choice(['thermal', 'dephasing'])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gates(case, seed):
    """The first case['gates'] gates of the workload, u3 and cx only."""
    n, count = case['n'], case['gates']
    kind = case['circuit']
    if kind == 'random':
        return workloads.random_u3_cx(n, count, seed)
    if kind == 'local':
        return workloads.local_u3_cx(n, count, seed)
    layers = 1 + count // n
    gates = workloads.matching_layers(n, layers, seed) if kind == 'matching' \
        else [g for g in workloads.brickwork_qft(n, layers, seed) if g[0] in ('u3', 'cx')]
    return gates[:count]


def _memory(case):
    return {'none': None, 'thermal': THERMAL, 'dephasing': DEPHASING}[case['memory']]


def _noise_after(case, i):
    return case['memory'] != 'none' and (i + 1) % case['every'] == 0


def _program(case, gates):
    n, mem = case['n'], _memory(case)
    if case['path'] == 'plain':
        prog = fusion.Program(n)
        for i, gate in enumerate(gates):
            for g in fusion.noisy_gates([gate], case['depol']):
                fusion.add_block(prog, [g], list(g.qubits), [0])
            if _noise_after(case, i):
                prog.memory_noise(mem['decoherence'], mem['thermal'], mem['decay'])
        return prog
    noisy = []
    for i, gate in enumerate(gates):
        noisy += fusion.noisy_gates([gate], case['depol'])
        if _noise_after(case, i):
            R = fusion.ptm.memory_noise(mem['decoherence'], mem['thermal'], mem['decay'])
            noisy += [fusion.NoisyGate((q,), R, 'u3') for q in range(n)]
    cost = None
    if case['path'] == 'learned':
        cost = costmodel.default_model()
        cost.precision = case['precision']
    # lookahead and block size as the backend plans
    prog, _ = fusion.fused_program(noisy, n, fusion.KMAX[case['path']], case['path'], cost,
                                   lookahead=fusion.LOOKAHEAD if n >= 15 else (), precision=case['precision'])
    return prog


class _DeviceVector:
    """The state's coefficient vector as a device array (no copy)."""

    def __init__(self, st):
        ptr = native.ctypes.c_void_p()
        native.check(st.lib.dm_device_ptr(st.h, native.ctypes.byref(ptr)), 'dm_device_ptr')
        self.st = st  # the buffer lives as long as the view
        self.__cuda_array_interface__ = {'shape': (st.size,), 'strides': None, 'version': 2,
                                         'typestr': '<f4' if st.dtype == native.FP32 else '<f8',
                                         'data': (ptr.value, False)}


def _view(st):
    return torch.as_tensor(_DeviceVector(st), device='cuda')


def _unit(seed):
    v = np.random.default_rng(seed + 17).normal(size=3)
    return v / np.linalg.norm(v)


def _measured(case, seed):
    return sorted(int(q) for q in np.random.default_rng(seed + 29).choice(case['n'], case['measured'], replace=False))


def _batch_specs(case, seed):
    """(n, gates, decay_rate, depol_rate) per circuit, as workloads.batch; the
    widths and depths belong to the case, the gates and rates to the seed."""
    shape, rng = np.random.default_rng(case['count']), np.random.default_rng(seed)
    out = []
    for i in range(case['count']):
        n = int(shape.integers(case['nlo'], case['nhi'] + 1))
        depth = int(shape.integers(case['dlo'], case['dhi'] + 1))
        decay, depol = (math.exp(x) for x in rng.uniform(math.log(1e-4), math.log(1e-2), 2))
        out.append((n, workloads.random_u3_cx(n, depth, int(rng.integers(1 << 31))), decay, depol))
    return out


def _readout_gates(case, seed):
    return workloads.local_u3_cx(case['n'], 2 * case['n'], seed)


def prepare(case, seed):
    kind = case['kind']
    if kind == 'circuit':
        st = native.DeviceState(case['n'], case['precision'])
        prog = _program(case, _gates(case, seed))
        prog.compile()
        return {'kind': kind, 'st': st, 'prog': prog, 'zero': np.tile([1.0, 0.0, 0.0, 1.0], case['n']),
                'qubits': list(range(case['n'])), 'vector': _view(st)}
    if kind == 'execute':
        mem = _memory(case)
        qc = workloads.to_circuit(case['n'], _gates(case, seed), barrier_after_each=True, measure=('ensemble', 'Z'))
        opts = {'decay_factor': mem['decay'], 'decoherence_factor': mem['decoherence'],
                'thermal_factor': mem['thermal'], 'depolarization_factor': 0.98, 'fusion': case['fusion'],
                'precision': case['precision'], 'compute_densitymatrix': True}
        return {'kind': kind, 'qc': qc, 'backend': BasicAer.get_backend('dm_simulator'), 'opts': opts}
    if kind == 'batch':
        b = batch.from_workload(_batch_specs(case, seed), case['precision'], lds_max_qubits=case['lds_max'],
                                lds_threads=case['threads'])
        return {'kind': kind, 'batch': b}
    n = case['n']
    states = []
    for precision, depol in ((case['precision'], 1e-3), (case['other'], 2e-3)):
        st = native.DeviceState(n, precision)
        v = _simulate(n, _readout_gates(case, seed), depol, None, 0)
        _view(st).copy_(v)
        states.append(st)
        del v
    return {'kind': kind, 'st': states[0], 'other': states[1], 'n': n, 'basis': case['basis'],
            'measured': _measured(case, seed), 'nvec': _unit(seed), 'dense': case['dense']}


def run(state):
    kind = state['kind']
    if kind == 'circuit':
        st = state['st']
        st.init_product(state['zero'], 0.5 ** st.n)
        state['prog'].run(st)
        return {'probabilities': st.probabilities(state['qubits'], 'Z'), 'coefficients': state['vector']}
    if kind == 'execute':
        data = execute(state['qc'], state['backend'], **state['opts']).result()['results'][0]['data']
        return {'ensemble': np.array(list(data['ensemble_probability'].values())),
                'densitymatrix': data['densitymatrix'], 'coeffmatrix': data['coeffmatrix']}
    if kind == 'batch':
        probs, _, _ = state['batch'].run(True)
        return {'probabilities': np.concatenate(probs)}
    st = state['st']
    out = {'ensemble': st.probabilities(list(range(state['n'])), 'Z', 0.99),
           'partial': st.probabilities(state['measured'], state['basis'], 0.99, state['nvec']),
           'trace_purity': np.array(st.trace_purity())}
    c = st.compare(state['other'])
    out['compare'] = np.array([c['max_abs_diff'], c['dot'], c['norm2_self'], c['norm2_other']])
    if state['dense']:
        out['densitymatrix'] = st.to_dense()
        out['coeffmatrix'] = st.download()
    return out


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------

def _gate_flops(n, u3, cx, levels):
    """A U3 with its channel: a 3x3 map on the X, Y, Z components (15 flops on
    3/4 of the coefficients, per group of four); a CX: one scale each; a
    memory-noise level: the product of the per-qubit factors, one scale and
    one feed per qubit's Z component."""
    N = 4.0 ** n
    return N * (u3 * 15 / 4 + cx + levels * (1 + n / 2))


def work(case):
    kind = case['kind']
    if kind == 'batch':
        byts = flops = 0.0
        for n in range(case['nlo'], case['nhi'] + 1):
            c = case['count'] / (case['nhi'] - case['nlo'] + 1)
            d = 0.5 * (case['dlo'] + case['dhi'])
            byts += c * (2 ** n * 8 + d * 100)
            flops += c * _gate_flops(n, 0.7 * d, 0.3 * d, d)
        return {'bytes': byts, 'flops': flops}
    n = case['n']
    N = 4.0 ** n
    s = 8 if case.get('precision') == 'fp64' else 4
    if kind == 'readout':
        so = 8 if case['other'] == 'fp64' else 4
        return {'bytes': N * (s + so) + (24.0 * N if case['dense'] else 0.0) + 2 ** n * 8, 'flops': 8.0 * N}
    u3 = 0.65 * case['gates']
    cx = case['gates'] - u3
    if kind == 'execute':
        return {'bytes': N * (s + 24.0), 'flops': _gate_flops(n, u3, cx, case['gates'] + 1)}
    levels = case['gates'] // case['every'] if case['every'] else 0
    # the state is written once; the initial state is a product state
    return {'bytes': N * s + 2 ** n * 8, 'flops': _gate_flops(n, u3, cx, levels)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _rotation(pair, angle):
    R = np.eye(4)
    i, j = pair
    R[i, i] = R[j, j] = math.cos(angle)
    R[i, j], R[j, i] = -math.sin(angle), math.sin(angle)
    return R


def _u3(theta, phi, lam):
    return _rotation((1, 2), phi) @ _rotation((3, 1), theta) @ _rotation((1, 2), lam)


def _digit(v, p):
    """The four components along position p, as views."""
    x = v.view(-1, 4, 4 ** p)
    return [x[:, c] for c in range(4)]


def _apply_1q(v, p, R):
    x = _digit(v, p)
    new = []
    for r in (1, 2, 3):
        acc = x[1] * R[r, 1]
        acc.add_(x[2], alpha=R[r, 2]).add_(x[3], alpha=R[r, 3])
        if R[r, 0] != 0.0:
            acc.add_(x[0], alpha=R[r, 0])
        new.append(acc)
    for r in (1, 2, 3):
        x[r].copy_(new[r - 1])


# CX conjugation of Pauli pairs (control, target): source of each moved pair
_CX = [((0, 2), (3, 2), 1), ((3, 2), (0, 2), 1), ((0, 3), (3, 3), 1), ((3, 3), (0, 3), 1), ((1, 0), (1, 1), 1),
       ((1, 1), (1, 0), 1), ((1, 2), (2, 3), 1), ((2, 3), (1, 2), 1), ((1, 3), (2, 2), -1), ((2, 2), (1, 3), -1),
       ((2, 0), (2, 1), 1), ((2, 1), (2, 0), 1)]


def _apply_cx(v, pc, pt, keep):
    hi, lo = max(pc, pt), min(pc, pt)
    x = v.view(-1, 4, 4 ** (hi - lo - 1), 4, 4 ** lo)

    def part(c, t):
        return x[:, c, :, t] if pc > pt else x[:, t, :, c]

    moved = {dst: part(*src) * float(sign) for dst, src, sign in _CX}
    for dst, val in moved.items():
        part(*dst).copy_(val)
    if keep != 1.0:
        # depolarising each of the two qubits: keep per non-identity component
        for p in (pc, pt):
            v.view(-1, 4, 4 ** p)[:, 1:].mul_(keep)


def _apply_memory(v, n, mem):
    od = math.sqrt(mem['decay']) * mem['decoherence']
    feed = (1 - mem['decay']) * (2 * mem['thermal'] - 1)
    for p in range(n):
        x = _digit(v, p)
        x[1].mul_(od)
        x[2].mul_(od)
        x[3].mul_(mem['decay'])
        if feed:
            x[3].add_(x[0], alpha=feed)


def _zero(n, device):
    v = torch.full((1,), 0.5 ** n, dtype=torch.float64, device=device)
    one = torch.tensor([1.0, 0.0, 0.0, 1.0], dtype=torch.float64, device=device)
    for _ in range(n):
        v = torch.outer(v, one).reshape(-1)
    return v


def _simulate(n, gates, depol, mem, every, device=DEVICE):
    v = _zero(n, device)
    for i, (name, qs, prm) in enumerate(gates):
        if name == 'u3':
            R = _u3(*prm)
            R[1:] *= 1.0 - depol
            _apply_1q(v, n - 1 - qs[0], R)
        else:
            _apply_cx(v, n - 1 - qs[0], n - 1 - qs[1], 1.0 - depol)
        if mem is not None and (i + 1) % every == 0:
            _apply_memory(v, n, mem)
    return v


def _probabilities(v, n, qubits, basis='Z', err=1.0, nvec=None):
    """Outcome probabilities of the qubits (first one most significant)."""
    x = v.view([4] * n)
    x = x[tuple(slice(None) if q in qubits else 0 for q in range(n))]
    vec = {'X': (1, 0, 0), 'Y': (0, 1, 0), 'Z': (0, 0, 1)}.get(basis)
    e = err * np.asarray(nvec if basis == 'N' else vec, dtype=float)
    for _ in qubits:  # contract the leading digit, append the outcome bit
        m = x[1] * e[0] + x[2] * e[1] + x[3] * e[2]
        x = torch.stack([x[0] + m, x[0] - m], dim=-1)
    return (x.reshape(-1) * 2.0 ** (n - len(qubits))).cpu().numpy()


def _dense(v, n):
    """Row-major density matrix: per qubit I+Z, X-iY / X+iY, I-Z."""
    x = v.to(torch.complex128)
    for _ in range(n):  # leading Pauli digit -> trailing (row, column) bits
        x = x.view(4, -1)
        x = torch.stack([x[0] + x[3], x[1] - 1j * x[2], x[1] + 1j * x[2], x[0] - x[3]], dim=-1).reshape(-1)
    x = x.cpu().numpy().reshape([2] * (2 * n))
    return np.ascontiguousarray(x.transpose([2 * q for q in range(n)] + [2 * q + 1 for q in range(n)])
                                .reshape(2 ** n, 2 ** n))


def exact(case, seed):
    kind = case['kind']
    if kind == 'circuit':
        n, mem = case['n'], _memory(case)
        levels = case['gates'] // case['every'] if mem else 0
        if 4.0 ** n * (case['gates'] + 0.5 * n * levels) * 1.3e-11 > 12.0:
            return None
        v = _simulate(n, _gates(case, seed), case['depol'], mem, case['every'])
        return {'probabilities': _probabilities(v, n, list(range(n))), 'coefficients': v}
    if kind == 'execute':
        n, mem = case['n'], _memory(case)
        v = _simulate(n, _gates(case, seed), 0.0, mem, 1)
        probs = _probabilities(v, n, list(range(n)), 'Z', 0.98)
        _apply_memory(v, n, mem)  # the measurement's own level ends with memory noise
        return {'ensemble': probs, 'densitymatrix': _dense(v, n), 'coeffmatrix': v.cpu().numpy()}
    if kind == 'batch':
        specs = _batch_specs(case, seed)
        if sum(len(g) * (3 + n) * max(1e-5, 4.0 ** n * 1e-9) for n, g, _, _ in specs) > 12.0:
            return None
        out = []
        for n, gates, decay, depol in specs:
            mem = {'decay': 1.0 - decay, 'decoherence': 1.0, 'thermal': 1.0}
            v = _simulate(n, gates, 0.0, mem, 1, 'cpu')
            out.append(_probabilities(v, n, list(range(n)), 'Z', 1.0 - depol))
        return {'probabilities': np.concatenate(out)}
    n = case['n']
    store = {'fp64': torch.float64, 'fp32': torch.float32}
    v, o = (_simulate(n, _readout_gates(case, seed), d, None, 0).to(store[p]).double()
            for p, d in ((case['precision'], 1e-3), (case['other'], 2e-3)))
    dot = [float(torch.dot(a, b)) for a, b in ((v, v), (v, o), (o, o))]
    out = {'ensemble': _probabilities(v, n, list(range(n)), 'Z', 0.99),
           'partial': _probabilities(v, n, _measured(case, seed), case['basis'], 0.99, _unit(seed)),
           'trace_purity': np.array([float(v[0]) * 2.0 ** n, dot[0] * 2.0 ** n]),
           'compare': np.array([float((v - o).abs().max()), dot[1], dot[0], dot[2]])}
    if case['dense']:
        out['densitymatrix'] = _dense(v, n)
        out['coeffmatrix'] = v.cpu().numpy()
    return out
