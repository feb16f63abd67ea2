"""Batches above 300 MiB of states: groups of circuits in two and three chains
of streams, against the same circuits one batch each (one group, one stream)
and two of them against the CPU oracle.

The circuits of a case have the same gates on the same qubits and differ in
their angles and noise rates, so that every group takes the launches of a
single circuit: the launch count says how many groups there were.  FP32
results do not depend on the grouping; FP64 to 1e-13, the oracle's tolerances
1e-12 (FP64) and 2e-5 (FP32) as for any batch.
"""
import numpy as np
import pytest

from dmsim import assemble, batch, native, workloads
from oracle import refsim

pytestmark = pytest.mark.gpu


def oracle_probs(n, gates, decay_rate, depol_rate):
    qc = workloads.to_circuit(n, gates, barrier_after_each=True, measure=('ensemble', 'Z'))
    exp = assemble(qc).experiments[0]
    data, _, _ = refsim.run_experiment(exp.instructions, n, {
        'decay_factor': 1.0 - decay_rate, 'depolarization_factor': 1.0 - depol_rate,
        'compute_densitymatrix': False})
    return np.array(list(data['ensemble_probability'].values()))


def alike(n, ngates, count, seed):
    """`count` circuits of the same gates and qubits."""
    rng = np.random.default_rng(seed)
    shape = workloads.random_u3_cx(n, ngates, seed, p_u3=0.6)
    out = []
    for _ in range(count):
        gates = [(name, qs, tuple(float(x) for x in rng.uniform(0, 2 * np.pi, 3)) if prm else ())
                 for name, qs, prm in shape]
        decay, depol = (float(x) for x in rng.uniform(1e-3, 1e-2, 2))
        out.append((n, gates, decay, depol))
    return out


def eager_work():
    """Kernels of another handle between replays of a batch's graph."""
    st = native.DeviceState(8, 'fp64')
    st.init_product(np.tile([1.0, 0.0, 0.0, 1.0], 8), 0.5 ** 8)
    st.memory_noise(0.99, 0.8, 0.97)
    purity = st.trace_purity()[1]
    st.close()
    assert 0 < purity <= 1


# 16 MiB a state, groups of 66 MiB in three chains; 128 MiB a state, groups of
# 100 MiB (one circuit each) in two
@pytest.mark.parametrize('precision,n,count,groups', [('fp32', 11, 24, 6), ('fp32', 11, 21, 6), ('fp64', 12, 3, 3),
                                                      ('fp64', 12, 4, 4)])
def test_groups_in_chains_equal_single_batches(precision, n, count, groups):
    specs = alike(n, 5, count, 40 + count)
    want, launches = [], set()
    for spec in specs:
        b = batch.from_workload([spec], precision, lds_max_qubits=6, lds_threads=256)
        want.append(b.run(False)[0][0])
        launches.add(b.info()['launches'])
        b.close()
    assert len(launches) == 1
    b = batch.from_workload(specs, precision, lds_max_qubits=6, lds_threads=256)
    assert b.info()['launches'] == groups * launches.pop()
    for graph in (False, True, True, True):
        probs, us, ms = b.run(graph)
        assert np.all(us > 0) and ms > 0
        for got, ref in zip(probs, want):
            if precision == 'fp32':
                assert np.array_equal(got, ref)
            else:
                assert np.abs(got - ref).max() <= 1e-13
        eager_work()
    b.close()
    for i in (0, count - 1):
        assert np.abs(want[i] - oracle_probs(*specs[i])).max() <= (1e-12 if precision == 'fp64' else 2e-5)


@pytest.mark.parametrize('precision', ['fp32', 'fp64'])
def test_uneven_circuits_of_every_tier_in_chains(precision):
    """Widths 2-12 and 3-12 gates in one batch: circuits in one workgroup
    beside groups whose members end in different rounds, one of them larger
    than a group."""
    rng = np.random.default_rng(17)
    widths = [12, 12, 12, 11, 11, 11, 10, 10, 9, 8, 7, 7, 6, 5, 3, 2] + ([12, 12, 12] if precision == 'fp32' else [])
    specs = [(n, workloads.random_u3_cx(n, int(rng.integers(3, 13)), 100 + i), 2e-3 + 1e-4 * i, 5e-3)
             for i, n in enumerate(widths)]
    assert sum(4 ** n for n in widths if n > 7) * (4 if precision == 'fp32' else 8) > 300 << 20
    want = []
    for spec in specs:
        b = batch.from_workload([spec], precision, lds_max_qubits=7, lds_threads=256)
        want.append(b.run(False)[0][0])
        b.close()
    b = batch.from_workload(specs, precision, lds_max_qubits=7, lds_threads=256)
    for graph in (False, True, True, True):
        for got, ref in zip(b.run(graph)[0], want):
            if precision == 'fp32':
                assert np.array_equal(got, ref)
            else:
                assert np.abs(got - ref).max() <= 1e-13
        eager_work()
    b.close()
