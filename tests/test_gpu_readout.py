"""Read-outs against the oracle at the sizes where their kernels change:
probabilities around the digits one launch contracts (12 of two components,
6 of four), product states around the digits of the LDS table (6), and the
FP64 sums.  Tolerances: a probability is a sum of 2^m (4^m) FP64 products
contracted pairwise, at most 3 m roundings of values <= its largest partial
sum (1 for a state of unit trace); a product has n + 1 factors; a sum of N
squares accumulated in blocks is within sqrt(N) eps of the exact one."""
import numpy as np
import pytest

from dmsim import native

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


def mixed_state(rng, n):
    """A product of single-qubit states with random Bloch vectors, plus a
    traceless perturbation small enough to keep probabilities below 2."""
    vecs = np.concatenate([np.ones((n, 1)), rng.uniform(-0.5, 0.5, (n, 3))], axis=1)
    a = np.ones(1)
    for q in range(n):
        a = np.kron(a, vecs[q])
    a *= 2.0 ** -n
    p = rng.normal(size=a.size) * 4.0 ** -n
    p[0] = 0.0
    return a + p, vecs


def probabilities(a, n, qubits, basis, err, nvec):
    x = a.reshape(n * [4])
    x = x[tuple(slice(None) if q in qubits else 0 for q in range(n))]
    e = err * np.asarray({'X': (1, 0, 0), 'Y': (0, 1, 0), 'Z': (0, 0, 1)}.get(basis, nvec), dtype=float)
    for _ in qubits:
        m = x[1] * e[0] + x[2] * e[1] + x[3] * e[2]
        x = np.stack([x[0] + m, x[0] - m], axis=-1)
    return x.reshape(-1) * 2.0 ** (n - len(qubits))


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
@pytest.mark.parametrize('n', [1, 4, 6, 7, 11, 12, 13])
def test_probabilities_of_one_to_all_qubits(n, precision):
    rng = np.random.default_rng(n)
    a, _ = mixed_state(rng, n)
    if precision == 'fp32':
        a = a.astype(np.float32).astype(np.float64)
    nvec = rng.normal(size=3)
    nvec /= np.linalg.norm(nvec)
    st = native.DeviceState(n, precision)
    st.upload(a)
    for m in sorted({1, (n + 1) // 2, max(1, n - 1), n}):
        qubits = sorted(int(q) for q in rng.choice(n, m, replace=False))
        for basis in 'XYZN':
            if basis == 'N' and m > 8:
                continue
            got = st.probabilities(qubits, basis, 0.93, nvec)
            want = probabilities(a, n, qubits, basis, 0.93, nvec)
            assert got.shape == want.shape
            assert np.abs(got - want).max() <= 3 * m * EPS * 4, (n, m, basis)
    st.close()


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
@pytest.mark.parametrize('n', [1, 2, 4, 5, 6, 7, 9])
def test_product_states_and_diagonals(n, precision):
    rng = np.random.default_rng(20 + n)
    eps = EPS if precision == 'fp64' else 2.0 ** -24
    _, vecs = mixed_state(rng, n)
    tab = rng.uniform(0.5, 1.0, (n, 4))
    want, factor = np.full(1, 2.0 ** -n), np.ones(1)
    for q in range(n):
        want, factor = np.kron(want, vecs[q]), np.kron(factor, tab[q])
    st = native.DeviceState(n, precision)
    st.init_product(vecs.reshape(-1), 2.0 ** -n)
    got = st.download()
    assert np.all(np.abs(got - want) <= (n + 2) * eps * np.abs(want))
    st.apply_diag(tab.reshape(-1))
    assert np.all(np.abs(st.download() - want * factor) <= (2 * n + 5) * eps * np.abs(want))
    st.close()


@pytest.mark.parametrize('n', [1, 3, 6, 11])
@pytest.mark.parametrize('pa,pb', [('fp64', 'fp64'), ('fp64', 'fp32'), ('fp32', 'fp64'), ('fp32', 'fp32')])
def test_sums(n, pa, pb):
    rng = np.random.default_rng(n)
    store = {'fp64': np.float64, 'fp32': np.float32}
    a = rng.normal(size=4 ** n).astype(store[pa]).astype(np.float64)
    b = rng.normal(size=4 ** n).astype(store[pb]).astype(np.float64)
    sa, sb = native.DeviceState(n, pa), native.DeviceState(n, pb)
    sa.upload(a)
    sb.upload(b)
    c = sa.compare(sb)
    tr, purity = sa.trace_purity()
    sa.close()
    sb.close()
    tol = 4 * np.sqrt(a.size) * EPS
    assert c['max_abs_diff'] == np.abs(a - b).max()
    aa, bb = np.dot(a, a), np.dot(b, b)
    assert abs(c['dot'] - np.dot(a, b)) <= tol * np.sqrt(aa * bb)
    assert abs(c['norm2_self'] - aa) <= tol * aa and abs(c['norm2_other'] - bb) <= tol * bb
    assert abs(purity - aa * 2.0 ** n) <= tol * aa * 2.0 ** n and tr == a[0] * 2.0 ** n


@pytest.mark.parametrize('n,pa,pb', [(n, pa, pb) for n in (8, 9, 10) for pa in ('fp64', 'fp32') for pb in ('fp64', 'fp32')]
                         + [(12, 'fp64', 'fp64'), (12, 'fp32', 'fp64')])
def test_sums_where_the_partials_move_to_the_device(n, pa, pb):
    """Up to 256 workgroups (8 qubits FP64 against FP64, 9 otherwise) the host
    adds their partials, above a kernel; 12 qubits: more packs than the
    workgroups take at once."""
    test_sums(n, pa, pb)


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
@pytest.mark.parametrize('n', [10, 11, 12, 13])
def test_product_states_and_diagonals_where_the_tables_change(n, precision):
    """Tables of 4^5 coefficients up to 10 qubits, of 4^6 above, and FP64
    diagonals without one from 12 (tolerances as above)."""
    test_product_states_and_diagonals(n, precision)


@pytest.mark.parametrize('n,precision', [(14, 'fp64'), (15, 'fp32'), (16, 'fp32')])
def test_probabilities_of_13_to_16_qubits(n, precision):
    """More than 12 two-component digits: 1-4 leading ones are contracted in
    registers.  A product state's probabilities are products of (1 +- err
    b_q) / 2, b_q another one for each qubit, so that a wrong digit order or
    column shows.  A coefficient has n + 1 factors, rounded to the storage
    type, and a sum of 2^m of them at most prod (1 + err |b_q|) 2^-m."""
    rng = np.random.default_rng(n)
    eps = EPS if precision == 'fp64' else 2.0 ** -24
    vecs = np.concatenate([np.ones((n, 1)), rng.uniform(0.1, 0.9, (n, 3)) * rng.choice([-1, 1], (n, 3))], axis=1)
    st = native.DeviceState(n, precision)
    st.init_product(vecs.reshape(-1), 2.0 ** -n)
    for m in range(13, n + 1):
        for basis, comp in (('X', 1), ('Z', 3)):
            qubits = sorted(int(q) for q in rng.choice(n, m, replace=False))
            want, top = np.ones(1), 1.0
            for q in qubits:
                b = 0.93 * vecs[q, comp]
                want = np.kron(want, [(1 + b) / 2, (1 - b) / 2])
                top *= (1 + abs(b)) / 2
            got = st.probabilities(qubits, basis, 0.93)
            assert got.shape == want.shape
            assert np.abs(got - want).max() <= ((n + 2) * eps + 6 * m * EPS) * top, (m, basis)
    st.close()
