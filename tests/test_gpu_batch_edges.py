"""Batch engine at the edges of its tiles: states below the four register
qubits, exactly one tile, one and two qubits more, for each tile size, with
every observable and shots read from resident and streamed states."""
import numpy as np
import pytest

from conftest import random_gate_list

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(0, 1e-12), (1, 2e-5)])
@pytest.mark.parametrize("tile_bits", [8, 9, 12])
def test_observables_and_shots_vs_oracle(eng, oracle, tile_bits, prec, tol):
    rng = np.random.default_rng(tile_bits)
    circuits = [{"n": n, "gates": random_gate_list(n, 40, rng), "precision": prec, "observables": 7,
                 "draws": rng.uniform(size=40)}
                for n in (1, 2, 3, 4, 5, tile_bits - 1, tile_bits, tile_bits + 1, tile_bits + 2)]
    b = eng.Batch()
    try:
        b.set_config(tile_bits=tile_bits)
        res = b.run(circuits)
    finally:
        b.free()
    for c, r in zip(circuits, res):
        n = c["n"]
        a = oracle.run(n, c["gates"])
        assert abs(r.norm - 1.0) < tol, n
        assert np.max(np.abs(r.expect_z - oracle.expect_z_all(n, a))) < tol, n
        if n > 1:
            zz = [oracle.correlation_zz(n, a, q, q + 1) for q in range(n - 1)]
            assert np.max(np.abs(r.zz_chain - zz)) < tol, n
        assert np.max(np.abs(r.expect_x - [oracle.expect_x(n, a, q) for q in range(n)])) < tol, n
        if prec == 0:
            assert r.outcomes.tolist() == [oracle.measure_all_outcome(n, a, u) for u in c["draws"]], n
        else:
            cdf = np.cumsum(np.abs(a) ** 2)   # outcome within rounding of the draw's place
            out = r.outcomes.astype(np.int64)
            assert np.all(cdf[out] > c["draws"] - 1e-4), n
            assert np.all(cdf[out] - np.abs(a[out]) ** 2 < c["draws"] + 1e-4), n
