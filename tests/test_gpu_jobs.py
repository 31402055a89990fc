"""Jobs around the choice between rotation passes and one kernel per gate:
states under the four register qubits, one gate and few, one tile and more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 4, 5, 12, 13, 17])
@pytest.mark.parametrize("gates", [1, 2, 5, 80])
def test_execute_ex_vs_oracle(eng, oracle, n, gates):
    rng = np.random.default_rng(100 * n + gates)
    rows, j = [], eng.Job(n)
    for _ in range(gates):
        t = int(rng.integers(0, 14))
        a, b = (int(q) for q in rng.permutation(n)[:2])
        th = float(rng.uniform(-7, 7))
        rows.append((t, a, b if t > 9 else -1, -1, th if t in (7, 8, 9) else 0.0))
        j.add_gate(t, a, b if t > 9 else -1, th if t in (7, 8, 9) else None)
    j.set_num_shots(300).set_num_workers(3).set_rng_seed(5)
    a = oracle.run(n, rows)
    r = j.execute_ex(amplitudes=True, probabilities=True, expect_z=True)
    assert np.max(np.abs(r.amplitudes - a)) < 1e-12
    assert np.max(np.abs(r.probabilities - np.abs(a) ** 2)) < 1e-12
    assert np.max(np.abs(r.expect_z - oracle.expect_z_all(n, a))) < 1e-12
    cdf = np.cumsum(np.abs(a) ** 2)
    out = np.asarray(r.outcomes, np.int64)
    assert np.array_equal(np.asarray(j.execute().outcomes), out)
    assert np.all(np.abs(a[out]) > 0) and cdf[out].max() <= 1 + 1e-12
    r = j.execute_ex(precision=eng.C64, amplitudes=True, skip_shots=True)
    assert np.max(np.abs(r.amplitudes - a)) < 2e-5


def test_results_outlive_each_other(eng):
    j = eng.Job(18)   # 4 MiB of amplitudes
    j.add_gate(4, 0)
    first = j.execute_ex(amplitudes=True, probabilities=True, skip_shots=True)
    a, p = first.amplitudes, first.probabilities
    del first
    for _ in range(3):
        j.execute_ex(amplitudes=True, probabilities=True, skip_shots=True)
    want = np.zeros(1 << 18)
    want[:2] = 0.5
    assert np.max(np.abs(p - want)) < 1e-15 and np.max(np.abs(np.abs(a) ** 2 - want)) < 1e-15
    a[0] = 0.0   # the array is the caller's own
    assert a[0] == 0.0
