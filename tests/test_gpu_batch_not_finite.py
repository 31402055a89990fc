"""Batch circuits with a parameter that is not finite: NaN where the gate acts
and nowhere else (as one kernel per gate and the oracle have it), the circuits
beside them untouched, and parameters that a gate does not read without effect."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")
# four equal amplitudes, then the gate; the last X moves NaN to the other value of qubit 2
TAILS = {
    "crx": [(19, 1, 2, -1, NAN)], "cphase": [(18, 0, 2, -1, INF)], "crz": [(21, 1, 2, -1, NAN), (4, 0, -1, -1, 0.0)],
    "phase": [(16, 2, -1, -1, -INF), (1, 2, -1, -1, 0.0)], "u3": [(17, 2, -1, -1, 0.0, NAN, 0.3), (10, 1, 0, -1, 0.0)],
    "cry": [(20, 0, 2, -1, INF), (1, 2, -1, -1, 0.0)], "all": [(8, 1, -1, -1, NAN)],
}


@pytest.mark.parametrize("n", [3, 9, 13])
@pytest.mark.parametrize("prec", [0, 1])
def test_not_finite_parameters_stay_where_they_act(eng, oracle, n, prec):
    draws = np.array([0.1, 0.3, 0.6, 0.9])
    head = [(4, 0, -1, -1, 0.0), (4, 1, -1, -1, 0.0)]
    pauli = [(1.0, "Z" + "I" * (n - 1)), (0.5, "IXI" + "I" * (n - 3))]
    def circuit(gates):
        return {"n": n, "gates": gates, "precision": prec, "observables": 7, "draws": draws, "pauli": pauli}
    finite = circuit(head + [(8, 2, -1, -1, 0.4), (10, 2, 1, -1, 0.0)])
    b = eng.Batch()
    try:
        alone = b.run([finite])[0]
        junk = b.run([circuit([(4, 0, -1, -1, NAN, INF, NAN), (4, 1, -1, -1, 0.0, NAN, 0.0), (8, 2, -1, -1, 0.4, NAN, INF),
                               (10, 2, 1, -1, INF)])])[0]
        assert junk.expect_z.tobytes() == alone.expect_z.tobytes() and junk.outcomes.tolist() == alone.outcomes.tolist()
        for name, tail in TAILS.items():
            first, bad, last = b.run([finite, circuit(head + tail), finite])
            a = oracle.run(n, head + tail)
            assert np.isnan(a).any(), name
            for r in (first, last):
                assert r.expect_z.tobytes() == alone.expect_z.tobytes() and r.norm == alone.norm, name
                assert r.outcomes.tolist() == alone.outcomes.tolist(), name
            assert np.isnan(bad.norm), name
            assert np.allclose(bad.expect_z, oracle.expect_z_all(n, a), rtol=0, atol=1e-5, equal_nan=True), name
            assert np.isnan(bad.zz_chain).all() and np.isnan(bad.expect_x).all() and np.isnan(bad.pauli_expect).all(), name
            assert bad.outcomes.tolist() == [oracle.measure_all_outcome(n, a, u) for u in draws], name
    finally:
        b.free()
