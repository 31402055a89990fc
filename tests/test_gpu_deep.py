"""Circuits of thousands of rotations in one pass (stored values are rescaled
on the way): blocked runs, jobs and batches against the oracle.

Tolerance: eight ulps of the norm a gate, both sides together."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def layers(n, depth, rng):
    """Hadamards (n = 10: random rotations) and CNOT brickwork on min(n, 12) qubits, then the rest joined."""
    rows, m = [], min(n, 12)
    for _ in range(depth):
        rows += [(int(rng.integers(7, 10)), q, -1, -1, float(rng.uniform(0, 6.2))) if n == 10 else (4, q, -1, -1, 0.0)
                 for q in range(m)]
        rows += [(10, q + 1, q, -1, 0.0) for o in (0, 1) for q in range(o, m - 1, 2)]
    for q in range(m, n):
        rows += [(4, q, -1, -1, 0.0), (10, q, q - m, -1, 0.0), (8, q - m, -1, -1, 0.3)]
    return rows


@pytest.mark.parametrize("n,depth", [(4, 760), (10, 1200), (12, 260), (14, 260)])
def test_deep_circuits_vs_oracle(eng, oracle, n, depth):
    g = layers(n, depth, np.random.default_rng(n))
    a = oracle.run(n, g)
    z = oracle.expect_z_all(n, a)
    job = eng.Job(n)
    for t, q, c, _, th in g:
        job.add_gate(t, q, c, th if t in (7, 8, 9) else None)
    b = eng.Batch()
    try:
        for prec, tol in ((eng.C128, len(g) * 2.0 ** -50), (eng.C64, len(g) * 2.0 ** -21)):
            with eng.StateVector(n, prec) as sv:
                got = sv.apply(g, blocked=True).amplitudes()
            assert np.linalg.norm(got - a) < tol
            r = job.execute_ex(precision=prec, amplitudes=True, expect_z=True, skip_shots=True)
            assert np.linalg.norm(r.amplitudes - a) < tol and np.max(np.abs(r.expect_z - z)) < 2 * tol
            r = b.run([{"n": n, "gates": g, "precision": prec, "observables": 1}])[0]
            assert abs(r.norm - 1.0) < 2 * tol and np.max(np.abs(r.expect_z - z)) < 2 * tol
    finally:
        b.free()
