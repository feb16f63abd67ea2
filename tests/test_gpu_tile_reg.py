"""Register-resident fused passes against the oracle.

Passes of single-qubit maps and CX gates take the register-resident kernel
from 12 qubits up, and FP64 passes of many operations from 7.  The cases cover
every place of the operands in the tile (load and store layouts, the digits
that lie across lanes, tiles of 5-7 digits completed to 7), unital, general
and diagonal maps, plain CX and CX with separable and general pair scales,
and the first and last digits of the register.
Tolerance: an output coefficient passes through at most one operation per
member, each a sum of at most 4 products of magnitude <= the state's largest
coefficient times the map's row norm (<= 2 here, kept below 1 on average by
the maps' contraction), so max|da| <= members * 8 eps * max over time of
max|a|, taken from the oracle's own states.
"""
import numpy as np
import pytest

from dmsim import native, ptm
from dmsim.program import Program
from oracle import refsim

pytestmark = pytest.mark.gpu

EPS = {'fp64': 2.0 ** -53, 'fp32': 2.0 ** -24}


def oracle_1q(a, n, q, R4):
    x = a.reshape(4 ** q, 4, 4 ** (n - q - 1))
    return np.einsum('ij,ajb->aib', R4, x).reshape(-1)


def oracle_cx(a, n, c, t, scale):
    x = refsim.apply_cx(a.copy().reshape(n * [4]), c, t, [1.0, 0.0], n)  # updates its argument
    if scale is not None:
        x = np.moveaxis(x, (c, t), (0, 1))
        x = np.asarray(scale).reshape(4, 4)[(...,) + (None,) * (n - 2)] * x
        x = np.moveaxis(x, (0, 1), (c, t))
    return np.ascontiguousarray(x).reshape(-1)


def random_map(rng, kind):
    R = np.eye(4)
    th, ph, la = rng.uniform(0, 2 * np.pi, 3)
    if kind != 'diag':
        R = ptm.gate_ptm('u3', [th, ph, la])
    R = ptm.depolarizing1(rng.uniform(0, 0.1)) @ R
    if kind == 'general':
        R = ptm.memory_noise(0.9, 0.8, 0.7) @ R
    return R


def random_scale(rng, kind):
    if kind == 'none':
        return None
    a, b = (np.concatenate([[1.0], rng.uniform(0.5, 1.0, 3)]) for _ in range(2))
    s = np.outer(a, b).reshape(16)
    if kind == 'general':
        s = rng.uniform(0.5, 1.0, 16)
        s[0] = 1.0
    return s


def check(n, m, qubits, members, precision, seed):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=4 ** n) * 2.0 ** -n
    a[0] = 2.0 ** -n
    if precision == 'fp32':
        a = a.astype(np.float32).astype(np.float64)
    want, top, sub = a, np.abs(a).max(), []
    for _ in range(members):
        if rng.random() < 0.5:
            q = int(rng.choice(qubits))
            R = random_map(rng, rng.choice(['unital', 'general', 'diag']))
            sub.append((native.SUB_1Q, [q], ptm.rows3(R)))
            want = oracle_1q(want, n, q, R)
        else:
            c, t = (int(x) for x in rng.choice(qubits, 2, replace=False))
            s = random_scale(rng, rng.choice(['none', 'separable', 'general']))
            sub.append((native.SUB_CX, [c, t], s))
            want = oracle_cx(want, n, c, t, s)
        top = max(top, np.abs(want).max())
    prog = Program(n)
    prog.fused(m, qubits, sub)
    st = native.DeviceState(n, precision)
    st.upload(a)
    prog.run(st)
    got = st.download()
    st.close()
    assert got[0] == 2.0 ** -n
    err = np.abs(got - want).max()
    assert err <= members * 8 * EPS[precision] * top, (n, m, qubits, seed, err, top)


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
@pytest.mark.parametrize('n,m,qubits', [
    (7, 7, [0, 1, 2]), (7, 7, [4, 5, 6]), (7, 6, [0, 6]), (8, 7, [0, 1, 2, 3]), (8, 5, [6, 7]), (8, 6, [1, 4, 7]),
    (9, 7, [0, 2, 4, 5]), (9, 6, [0, 1, 2]), (9, 7, [0, 1, 7, 8]),
])
def test_many_members_on_few_qubits(n, m, qubits, precision):
    for seed in range(4):
        check(n, m, qubits, 24 + 8 * seed, precision, 100 * n + seed)


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
@pytest.mark.parametrize('qubits,members', [([0, 1, 2, 3], 1), ([11], 3), ([0, 5, 10, 11], 9), ([8, 9, 10, 11], 14),
                                            ([0, 3, 6], 0)])
def test_every_pass_from_12_qubits(qubits, members, precision):
    if len(qubits) == 1:
        n = 12
        rng = np.random.default_rng(5)
        a = rng.normal(size=4 ** n) * 2.0 ** -n
        a[0] = 2.0 ** -n
        a = a.astype(np.float32).astype(np.float64)
        R = random_map(rng, 'general')
        prog = Program(n)
        prog.fused(6, qubits, [(native.SUB_1Q, qubits, ptm.rows3(R))] * members)
        st = native.DeviceState(n, precision)
        st.upload(a)
        prog.run(st)
        got = st.download()
        st.close()
        want = a
        for _ in range(members):
            want = oracle_1q(want, n, qubits[0], R)
        assert np.abs(got - want).max() <= members * 8 * EPS[precision] * np.abs(a).max()
        return
    check(12, 7, qubits, members, precision, 7)


def with_identity(sub, qubits):
    """The same operations and an identity two-qubit map, which the
    register-resident kernels leave to the tile-in-LDS form."""
    return sub + [(native.SUB_2Q, list(qubits[:2]), np.eye(16))]


@pytest.mark.parametrize('n,m,qubits', [(8, 7, [0, 2, 3, 7]), (9, 6, [0, 1, 4]), (12, 7, [0, 1, 10, 11]),
                                        (12, 6, [6, 7, 8]), (12, 7, [2, 4, 8, 10]), (12, 7, [8, 9, 10, 11])])
def test_fp32_passes_equal_the_lds_form_bit_for_bit(n, m, qubits):
    """FP32 keeps the order of operations: the state is the same whichever
    form ran."""
    rng = np.random.default_rng(n)
    sub = []
    for _ in range(40):
        if rng.random() < 0.5:
            R = random_map(rng, rng.choice(['unital', 'general', 'diag']))
            sub.append((native.SUB_1Q, [int(rng.choice(qubits))], ptm.rows3(R)))
        else:
            c, t = (int(x) for x in rng.choice(qubits, 2, replace=False))
            sub.append((native.SUB_CX, [c, t], random_scale(rng, rng.choice(['none', 'separable', 'general']))))
    a = rng.normal(size=4 ** n) * 2.0 ** -n
    got = []
    for ops in (sub, with_identity(sub, qubits)):
        prog = Program(n)
        prog.fused(m, qubits, ops)
        st = native.DeviceState(n, 'fp32')
        st.upload(a)
        prog.run(st)
        got.append(st.download())
        st.close()
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize('n,precision', [(13, 'fp64'), (14, 'fp32')])
def test_states_above_the_last_level_cache(n, precision):
    """Every tile is visited once: passes of single-qubit maps take a product
    state to the product of the mapped vectors (each coefficient a product of
    n + 1 factors on either side, and one sum of 4 products a map)."""
    rng = np.random.default_rng(n)
    vecs = np.concatenate([np.ones((n, 1)), rng.uniform(-0.5, 0.5, (n, 3))], axis=1)
    prog = Program(n)
    st = native.DeviceState(n, precision)
    st.init_product(vecs.reshape(-1), 2.0 ** -n)
    for qubits in ([0, 1, 2, 3], [n - 7, n - 6, n - 5, n - 4], [n - 4, n - 3, n - 2, n - 1], [0, 4, n - 1]):
        members = [(q, random_map(rng, 'general')) for _ in range(4) for q in qubits]
        prog.fused(7, qubits, [(native.SUB_1Q, [q], ptm.rows3(R)) for q, R in members])
        for q, R in members:
            vecs[q] = R @ vecs[q]
    prog.run(st)
    want = native.DeviceState(n, precision)
    want.init_product(vecs.reshape(-1), 2.0 ** -n)
    r = st.compare(want)
    st.close()
    want.close()
    assert r['max_abs_diff'] <= (60 * 8 + 2 * (n + 2)) * EPS[precision] * 2.0 ** -n


def small_circuit(rng, n, ngates, noise):
    """(Program, the oracle's probabilities) of a random circuit with memory
    noise after every gate, depolarising CX scales and a final measurement
    with retention 0.97."""
    prog = Program(n)
    a = refsim.initial_state(n).reshape(-1)
    for _ in range(ngates):
        if n == 1 or rng.random() < 0.6:
            q = int(rng.integers(n))
            R = random_map(rng, rng.choice(['unital', 'general', 'diag']))
            prog.one_qubit(q, R)
            a = oracle_1q(a, n, q, R)
        else:
            c, t = (int(x) for x in rng.choice(n, 2, replace=False))
            s = random_scale(rng, rng.choice(['none', 'separable', 'general']))
            prog.cx(c, t, s)
            a = oracle_cx(a, n, c, t, s)
        if noise is not None:
            prog.memory_noise(*noise)
            a = refsim.apply_memory_noise(a.copy().reshape(n * [4]), n, *noise).reshape(-1)
    x = a.reshape(n * [4])
    for _ in range(n):
        x = np.stack([x[0] + 0.97 * x[3], x[0] - 0.97 * x[3]], axis=-1)
    return prog, x.reshape(-1)


@pytest.mark.parametrize('noise', [None, (0.98, 0.8, 0.995), (0.98, 0.5, 1.0)])
@pytest.mark.parametrize('precision,tol', [('fp64', 1e-12), ('fp32', 2e-5)])
def test_whole_circuits_in_registers(precision, tol, noise):
    """Registers of 1-7 qubits, programs of 0-60 gates (the batch tests'
    tolerances: 1e-12 in FP64, 2e-5 in FP32)."""
    from dmsim import batch
    rng = np.random.default_rng(11)
    cases = [(n, *small_circuit(rng, n, g, noise)) for n in range(1, 8) for g in (0, 1, 7, 60)]
    b = batch.Batch([(n, prog, 0.97) for n, prog, _ in cases], precision, lds_max_qubits=7, lds_threads=256)
    for graph in (False, True, True):
        probs, us, _ = b.run(graph)
        assert np.all(us > 0)
        for (n, _, want), got in zip(cases, probs):
            assert np.max(np.abs(got - want)) <= tol, n
    b.close()


def test_fp32_whole_circuits_equal_the_lds_kernel_bit_for_bit():
    from dmsim import batch
    rng = np.random.default_rng(3)
    out = []
    circuits = [(n, small_circuit(rng, n, 40, (0.98, 0.8, 0.995))[0], 0.97) for n in range(2, 8)]
    for lds in (False, True):
        if lds:  # an identity two-qubit map: whole circuits in LDS
            for n, prog, _ in circuits:
                prog.two_qubit(0, 1, np.eye(16))
        b = batch.Batch(circuits, 'fp32', lds_max_qubits=7, lds_threads=256)
        out.append(np.concatenate(b.run(False)[0]))
        b.close()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize('n', [1, 2, 3, 5, 6, 7, 8, 10, 12])
@pytest.mark.parametrize('noise', [None, (0.98, 0.8, 0.995), (0.98, 0.5, 1.0)])
def test_fp64_runs_of_single_operations(n, noise):
    """Programs of single-qubit, CX and memory-noise operations, which an
    FP64 state runs as fused passes, against the oracle: runs of 2 to 30
    operations, broken by a diagonal operation that keeps its own kernel.
    Tolerance: each of the at most 30 (1 + n) maps rounds a coefficient by
    at most 8 eps of the largest one."""
    rng = np.random.default_rng(40 + n)
    for ngates in ((2, 9, 30) if n < 12 else (12,)):
        prog, _ = small_circuit(rng, n, ngates, noise)
        keep = rng.uniform(0.9, 1.0, (n, 4))
        keep[:, 0] = 1.0
        prog.diag(keep.reshape(-1))
        q = int(rng.integers(n))
        prog.one_qubit(q, ptm.memory_noise(0.9, 0.8, 0.7))
        st = native.DeviceState(n, 'fp64')
        a = rng.normal(size=4 ** n) * 2.0 ** -n
        a[0] = 2.0 ** -n
        st.upload(a)
        prog.run(st)
        arr, params = prog.compile()
        want = a
        for i in range(len(prog)):
            op, v = arr[i], params[arr[i].param:]
            if op.kind == native.OP_1Q:
                want = oracle_1q(want, n, op.qubits[0], np.vstack([[1.0, 0, 0, 0], v[:12].reshape(3, 4)]))
            elif op.kind in (native.OP_CX, native.OP_CX_SCALED):
                s = v[:16] if op.kind == native.OP_CX_SCALED else None
                want = oracle_cx(want, n, op.qubits[0], op.qubits[1], s)
            elif op.kind == native.OP_MEMORY_NOISE:
                want = refsim.apply_memory_noise(want.copy().reshape(n * [4]), n, *v[:3]).reshape(-1)
            else:
                x = want.reshape(n * [4])
                for p in range(n):
                    x = np.moveaxis(np.moveaxis(x, p, -1) * v[4 * p:4 * p + 4], -1, p)
                want = np.ascontiguousarray(x).reshape(-1)
        got = st.download()
        st.close()
        assert got[0] == 2.0 ** -n
        assert np.abs(got - want).max() <= 30 * (1 + n) * 8 * EPS['fp64'] * np.abs(a).max()


@pytest.mark.parametrize('n,m', [(5, 5), (6, 5), (6, 6)])
@pytest.mark.parametrize('dense', [False, True])
def test_fp64_fused_passes_join_the_run_of_a_small_register(n, m, dense):
    """Fused passes and single operations in one program of 5 or 6 qubits;
    `dense`: one pass holds a two-qubit map, which breaks the run.
    Tolerance: as the passes above, members * 8 eps * the largest
    coefficient."""
    rng = np.random.default_rng(10 * n + m + dense)
    a = rng.normal(size=4 ** n) * 2.0 ** -n
    a[0] = 2.0 ** -n
    want, members, prog = a, 0, Program(n)
    top = np.abs(a).max()
    for k in range(5):
        qubits = sorted({int(q) for q in rng.choice(n, m - 2, replace=False)} | {n - 1})
        sub = []
        for _ in range(int(rng.integers(0, 12))):
            if rng.random() < 0.5:
                q = int(rng.choice(qubits))
                R = random_map(rng, rng.choice(['unital', 'general', 'diag']))
                sub.append((native.SUB_1Q, [q], ptm.rows3(R)))
                want = oracle_1q(want, n, q, R)
            else:
                c, t = (int(x) for x in rng.choice(qubits, 2, replace=False))
                s = random_scale(rng, rng.choice(['none', 'separable', 'general']))
                sub.append((native.SUB_CX, [c, t], s))
                want = oracle_cx(want, n, c, t, s)
            top = max(top, np.abs(want).max())
        if dense and k == 2:
            sub = with_identity(sub, qubits)
        prog.fused(m, qubits, sub)
        q, R = int(rng.integers(n)), random_map(rng, 'general')
        prog.one_qubit(q, R)
        want = oracle_1q(want, n, q, R)
        top = max(top, np.abs(want).max())
        members += len(sub) + 1
    st = native.DeviceState(n, 'fp64')
    st.upload(a)
    prog.run(st)
    got = st.download()
    st.close()
    assert got[0] == 2.0 ** -n
    assert np.abs(got - want).max() <= members * 8 * EPS['fp64'] * top


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_program_images_of_every_size_and_in_turn(precision):
    """Images of a few hundred bytes to above 256 KiB, one program after the
    other on one handle without a wait between them, often enough for the
    uploads from pageable and from pinned memory, against the same programs
    each on a handle of its own: the same bit for bit."""
    n = 7
    rng = np.random.default_rng(8)
    progs = []
    for passes in (1, 4, 40, 700, 3, 41):  # about 0.4 KB a pass and more
        prog = Program(n)
        for _ in range(passes):
            c, t = (int(x) for x in rng.choice(n, 2, replace=False))
            prog.fused(7, [c, t], [(native.SUB_1Q, [c], ptm.rows3(random_map(rng, 'general'))),
                                   (native.SUB_CX, [c, t], random_scale(rng, 'general')),
                                   (native.SUB_1Q, [t], ptm.rows3(random_map(rng, 'unital')))])
        progs.append(prog)
    a = rng.normal(size=4 ** n) * 2.0 ** -n
    kept = native.DeviceState(n, precision)
    kept.upload(a)
    for _ in range(6):
        for prog in progs:
            prog.run(kept)
    got = kept.download()
    kept.close()
    for _ in range(6):
        for prog in progs:
            st = native.DeviceState(n, precision)
            st.upload(a)
            prog.run(st)
            a = st.download()
            st.close()
    assert np.array_equal(got, a)


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_whole_circuits_in_lds_of_all_widths(precision):
    """Circuits of 1-6 qubits that keep the LDS kernel (FP32; in FP64 those
    with a two-qubit map) are one launch, those of 7 another (in FP32 the
    register-resident one), each circuit as in a batch of its own."""
    from dmsim import batch
    rng = np.random.default_rng(5)
    circuits = []
    for n in (3, 1, 6, 7, 2, 5, 7, 4, 6):
        prog, _ = small_circuit(rng, n, 12, (0.98, 0.8, 0.995))
        if precision == 'fp64' and n > 1:
            prog.two_qubit(0, 1, np.eye(16))
        circuits.append((n, prog, 0.97))
    b = batch.Batch(circuits, precision, lds_max_qubits=7, lds_threads=256)
    assert b.info()['launches'] == (2 if precision == 'fp32' else 3)  # FP64: one qubit stays in registers
    for graph in (False, True, True):
        for circuit, got in zip(circuits, b.run(graph)[0]):
            one = batch.Batch([circuit], precision, lds_max_qubits=7, lds_threads=256)
            assert np.array_equal(one.run(False)[0][0], got)
            one.close()
    b.close()


@pytest.mark.parametrize('n,m,qubits,precision', [
    (13, 5, [0, 2, 3], 'fp64'), (13, 5, [0, 1, 2, 3], 'fp32'), (13, 5, [9, 12], 'fp64'), (13, 6, [1, 3, 5, 7], 'fp32'),
    (14, 5, [0, 1, 2, 3], 'fp32'), (14, 6, [0, 1, 2, 3], 'fp32'), (14, 6, [4, 6, 7, 12], 'fp32'),
    (14, 6, [3, 4, 5, 6], 'fp64'), (14, 5, [2, 13], 'fp64')])
def test_small_tiles_of_large_states(n, m, qubits, precision):
    """Passes whose tile is widened (5 digits from 13 qubits, FP32 6 digits of
    short runs from 14) or kept to four workgroups a CU, with two-qubit maps,
    against one kernel an operation.  Tolerance as above on either side."""
    rng = np.random.default_rng(n + m)
    vecs = np.concatenate([np.ones((n, 1)), rng.uniform(-0.5, 0.5, (n, 3))], axis=1)
    fused, plain = native.DeviceState(n, precision), native.DeviceState(n, precision)
    for st in (fused, plain):
        st.init_product(vecs.reshape(-1), 2.0 ** -n)
    sub, members = [], 9
    for i in range(members):
        c, t = (int(x) for x in rng.choice(qubits, 2, replace=False))
        if i % 3 == 0:
            R = random_map(rng, 'general')
            sub.append((native.SUB_1Q, [c], ptm.rows3(R)))
            plain.apply_1q(c, ptm.rows3(R))
        elif i % 3 == 1:
            s = random_scale(rng, 'general')
            sub.append((native.SUB_CX, [c, t], s))
            plain.apply_cx(c, t, s)
        else:
            R = ptm.cx_ptm((0.97, 0.02)) @ np.kron(random_map(rng, 'general'), random_map(rng, 'unital'))
            sub.append((native.SUB_2Q, [c, t], R))
            plain.apply_2q(c, t, R)
    prog = Program(n)
    prog.fused(m, qubits, sub)
    prog.run(fused)
    r = fused.compare(plain)
    fused.close()
    plain.close()
    # a sum of at most 16 products a two-qubit member
    assert r['max_abs_diff'] <= 2 * members * 32 * EPS[precision] * 2.0 ** -n
    assert r['norm2_self'] > 0


def random_members(rng, qubits, count):
    sub = []
    for _ in range(count):
        if rng.random() < 0.4:
            R = random_map(rng, rng.choice(['unital', 'general', 'diag']))
            sub.append((native.SUB_1Q, [int(rng.choice(qubits))], ptm.rows3(R)))
        else:
            c, t = (int(x) for x in rng.choice(qubits, 2, replace=False))
            sub.append((native.SUB_CX, [c, t], random_scale(rng, rng.choice(['none', 'separable', 'general']))))
    return sub


# FP32 passes in registers are those from 12 qubits (13: 256 MB, the largest
# state with plain accesses; 14: nontemporal, passes of 12 members and more),
# FP64 ones above the last-level cache from 13
@pytest.mark.parametrize('n,precision', [(12, 'fp32'), (13, 'fp32'), (14, 'fp32'), (13, 'fp64'), (14, 'fp64')])
def test_cx_passes_of_large_states_against_the_lds_form(n, precision):
    """Passes of maps, CX and scales on low, high and scattered digits, each
    state against the one that an identity two-qubit map in every pass keeps
    in LDS: FP32 bit for bit, FP64 to 8 eps a member and side."""
    rng = np.random.default_rng(60 + n)
    vecs = np.concatenate([np.ones((n, 1)), rng.uniform(-0.9, 0.9, (n, 3))], axis=1)
    reg, lds = Program(n), Program(n)
    members = 0
    for qubits in ([0, 1, 2, 3], [n - 4, n - 3, n - 2, n - 1], [0, 4, n - 5, n - 1], [n - 7, n - 6, n - 5, n - 4]):
        sub = random_members(rng, qubits, 40)
        members += len(sub)
        reg.fused(7, qubits, sub)
        lds.fused(7, qubits, with_identity(sub, qubits))
    a, b = native.DeviceState(n, precision), native.DeviceState(n, precision)
    for st, prog in ((a, reg), (b, lds)):
        st.init_product(vecs.reshape(-1), 2.0 ** -n)
        prog.run(st)
    r = a.compare(b)
    a.close()
    b.close()
    assert r['norm2_self'] > 4.0 ** -n
    assert r['max_abs_diff'] <= (0.0 if precision == 'fp32' else 2 * members * 8 * EPS['fp64'] * 2.0 ** -n)


def test_fp32_batch_passes_in_registers_equal_the_lds_form():
    """Batches of as many tiles as CUs take the register form at every width
    (8-10 qubits here), a state of that size by itself keeps the LDS form: the
    same coefficients, so that the probabilities differ by FP64 roundings
    only (an FP32 one would be 1e-10)."""
    from dmsim import batch
    rng = np.random.default_rng(9)
    circuits = []
    for n in (8, 9, 10, 10, 10, 10, 10):
        prog = Program(n)
        for _ in range(5):
            qubits = sorted(int(q) for q in rng.choice(n, 4, replace=False))
            prog.fused(6, qubits, random_members(rng, qubits, 16))
        circuits.append((n, prog, 0.97))
    b = batch.Batch(circuits, 'fp32', lds_max_qubits=6, lds_threads=256)
    got = b.run(False)[0]
    b.close()
    for (n, prog, err), probs in zip(circuits, got):
        st = native.DeviceState(n, 'fp32')
        st.init_product(np.tile([1.0, 0.0, 0.0, 1.0], n), 2.0 ** -n)
        prog.run(st)
        assert np.abs(probs - st.probabilities(list(range(n)), 'Z', err)).max() <= 3 * n * 2.0 ** -53
        st.close()


@pytest.mark.parametrize('n', [13, 14])
@pytest.mark.parametrize('noise', [None, (0.98, 0.8, 0.995)])
def test_fp64_runs_of_single_operations_above_the_last_level_cache(n, noise):
    """A program's run of single operations (fused passes, nontemporal, tiles
    handed to the XCDs in runs) against one call an operation.  Tolerance as
    for the smaller runs, on either side."""
    rng = np.random.default_rng(80 + n)
    vecs = np.concatenate([np.ones((n, 1)), rng.uniform(-0.5, 0.5, (n, 3))], axis=1)
    run, single = native.DeviceState(n, 'fp64'), native.DeviceState(n, 'fp64')
    for st in (run, single):
        st.init_product(vecs.reshape(-1), 2.0 ** -n)
    prog = Program(n)
    ops = 24
    for i in range(ops):
        if i % 2 == 0:
            q, R = int(rng.integers(n)), random_map(rng, 'general')
            prog.one_qubit(q, R)
            single.apply_1q(q, ptm.rows3(R))
        else:
            c, t = (int(x) for x in rng.choice(n, 2, replace=False))
            s = random_scale(rng, rng.choice(['none', 'separable', 'general']))
            prog.cx(c, t, s)
            single.apply_cx(c, t, s)
        if noise is not None and i % 8 == 7:
            prog.memory_noise(*noise)
            single.memory_noise(*noise)
    prog.run(run)
    r = run.compare(single)
    run.close()
    single.close()
    assert r['norm2_self'] > 4.0 ** -n
    assert r['max_abs_diff'] <= 2 * (ops + 3 * n) * 8 * EPS['fp64'] * 2.0 ** -n
