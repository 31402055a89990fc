"""Final sums of the reductions and of the outcome tables: sizes on both sides
of one 4096-amplitude tile, of one workgroup of partials and of the outcome
table's two summing kernels."""
import numpy as np
import pytest

from conftest import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 6, 8, 11, 12, 13, 21])
def test_norm_and_z_match_numpy(eng, n):
    a = random_state(n, np.random.default_rng(n)) * 1.5
    with eng.StateVector(n) as sv:
        sv.load(a)
        z, norm = sv.expect_z_all()
        p = np.abs(a) ** 2
        assert abs(norm - p.sum()) < 1e-12
        for q in range(n):
            assert abs(z[q] - (1.0 - 2.0 * p.reshape(-1, 2, 1 << q)[:, 1].sum())) < 1e-12
        assert abs(sv.expect_x(0) - 2.0 * np.sum(a[0::2].conj() * a[1::2]).real) < 1e-12


@pytest.mark.parametrize("n,k", [(13, 1), (17, 1), (18, 1), (18, 2), (20, 7), (12, 12)])
def test_outcome_sums_match_numpy(eng, n, k):
    a = random_state(n, np.random.default_rng(n + 100 * k))
    qubits = list(np.random.default_rng(k).permutation(n)[:k])
    out = np.zeros(1 << n, dtype=np.int64)
    for j, q in enumerate(qubits):
        out |= ((np.arange(1 << n) >> int(q)) & 1) << j
    p = np.bincount(out, np.abs(a) ** 2, minlength=1 << k)
    cum = np.cumsum(p)
    want = int(np.argmax(cum > 0.5))
    with eng.StateVector(n) as sv:
        sv.load(a)
        assert sv.measure_partial(qubits, 0.5) == want
        b = sv.amplitudes()
    keep = out == want
    assert not np.any(b[~keep])
    assert np.max(np.abs(b[keep] - a[keep] / np.sqrt(p[want]))) < 1e-12
