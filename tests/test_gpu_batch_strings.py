"""Pauli strings of a batch measured by workgroups of their own: the bits of
the persistent kernel's measurement and the oracle's values, for states below,
of and above one tile, and numbers of strings around one workgroup's eight."""
import numpy as np
import pytest

from conftest import random_gate_list

pytestmark = pytest.mark.gpu


def strings(n, k, rng):
    return [(float(rng.normal()), "".join(rng.choice(list("IXYZ"), size=n))) for _ in range(k)]


@pytest.mark.parametrize("prec,tol", [(0, 1e-12), (1, 2e-5)])
def test_strings_alone_and_beside_a_heavy_circuit(eng, oracle, prec, tol):
    rng = np.random.default_rng(7 + prec)
    # few enough to stay with the persistent kernel when alone
    light = [{"n": n, "gates": random_gate_list(n, 40, rng), "precision": prec, "pauli": strings(n, k, rng)}
             for n, k in ((1, 1), (4, 7), (7, 8), (9, 9), (11, 16), (12, 8), (13, 4), (14, 2))]
    heavy = [{"n": n, "gates": random_gate_list(n, 40, rng), "precision": p, "pauli": strings(n, k, rng)}
             for n, k, p in ((15, 33, 0), (12, 60, 1))]
    b = eng.Batch()
    try:
        alone = [b.run([c])[0].pauli_expect for c in light]
        for _ in range(3):   # launched, captured, replayed
            mixed = b.run(light + heavy)
            for c, a, r in zip(light, alone, mixed):
                assert r.pauli_expect.tobytes() == a.tobytes(), c["n"]
            for c, r in zip(light + heavy, mixed):
                a = oracle.run(c["n"], c["gates"])
                want = [oracle.expect_pauli(c["n"], a, s) for _, s in c["pauli"]]
                t = tol if c["precision"] == prec else 2e-5
                assert np.max(np.abs(r.pauli_expect - want)) < max(t, tol), c["n"]
    finally:
        b.free()
