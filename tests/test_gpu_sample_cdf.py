"""Shots through the cumulative table (eight per tile or more) and through the
per-shot scan of a tile: the oracle's outcomes from both, draws at and past
the ends among them."""
import numpy as np
import pytest

from conftest import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 7, 8, 11, 12, 13, 16])
def test_table_and_scan_give_the_oracles_outcomes(eng, oracle, n):
    rng = np.random.default_rng(n)
    a = random_state(n, rng)
    a[-1] = 0.0   # the last index with mass is another
    ends = [0.0, 1.0 - 2.0 ** -53, 1.0, 3.0]
    few = np.concatenate([rng.uniform(size=3), ends])
    many = np.concatenate([rng.uniform(size=8 * max(1, 1 << max(n - 12, 0)) + 5), ends])
    with eng.StateVector(n) as sv:
        sv.load(a)
        for u in (few, many):
            want = [oracle.measure_all_outcome(n, a, x) for x in u]
            assert np.asarray(sv.sample(u)).tolist() == want, len(u)
    with eng.StateVector(n, eng.C64) as sv:
        sv.load(a)
        got = sv.sample(many)
        one = np.concatenate([sv.sample(many[i:i + 5]) for i in range(0, len(many), 5)])
        assert np.asarray(got).tolist() == np.asarray(one).tolist()
