"""Few large circuits in a batch: their passes run over the whole chip, and
their results are those of the same circuits in a batch that keeps each on one
workgroup; empty circuits beside them, both precisions, and graph replays."""
import numpy as np
import pytest

from conftest import random_gate_list

pytestmark = pytest.mark.gpu


def circuits(rng, sizes, gates):
    return [{"n": n, "gates": random_gate_list(n, gates, rng) if k else [], "precision": k % 2, "observables": 7,
             "draws": rng.uniform(size=30)} for k, n in enumerate(sizes)]


@pytest.mark.parametrize("sizes", [[13, 13], [14, 17, 9, 18, 12, 16], [15, 20, 19]])
def test_spread_circuits(eng, oracle, sizes):
    rng = np.random.default_rng(sum(sizes))
    few = circuits(rng, sizes, 150)
    b = eng.Batch()
    try:
        for _ in range(3):   # launched, captured, replayed
            res = b.run(few)
            for c, r in zip(few, res):
                n, tol = c["n"], 1e-12 if c["precision"] == 0 else 2e-5
                a = oracle.run(n, c["gates"])
                assert abs(r.norm - 1.0) < tol
                assert np.max(np.abs(r.expect_z - oracle.expect_z_all(n, a))) < tol
                assert np.max(np.abs(r.expect_x - [oracle.expect_x(n, a, q) for q in range(n)])) < tol
                if c["precision"] == 0:
                    assert r.outcomes.tolist() == [oracle.measure_all_outcome(n, a, u) for u in c["draws"]]
        many = b.run(few + circuits(rng, [12] * 3000, 150))   # enough to keep each on its workgroup
        for r, m in zip(res, many):
            assert r.expect_z.tobytes() == m.expect_z.tobytes() and r.outcomes.tobytes() == m.outcomes.tobytes()
            assert r.expect_x.tobytes() == m.expect_x.tobytes() and r.norm == m.norm
    finally:
        b.free()
