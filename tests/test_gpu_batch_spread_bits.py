"""Passes of large circuits over the whole chip and on one workgroup: the same
bits.  Beside 260 circuits of 20 qubits the states pass 2^28 amplitudes, above
which no circuit gets a slot of its own, so each keeps to its workgroup; alone,
the longest circuit outlasts the spread passes by far at every size here."""
import numpy as np
import pytest

from conftest import random_gate_list

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[14, 14, 14], [14, 17, 9, 18, 12, 16], [15, 20, 19]])
def test_spread_and_one_workgroup_agree(eng, sizes):
    rng = np.random.default_rng(sum(sizes))
    few = [{"n": n, "gates": random_gate_list(n, 150, rng), "precision": p, "observables": 7,
            "draws": rng.uniform(size=30)} for n in sizes for p in (0, 1)]
    fill = [{"n": 20, "gates": [(4, 0)], "precision": 0, "observables": 0}] * 260
    b = eng.Batch()
    try:
        spread, alone = b.run(few), b.run(few + fill)
    finally:
        b.free()
    for c, r, s in zip(few, spread, alone):
        assert r.norm == s.norm, c["n"]
        for x, y in ((r.expect_z, s.expect_z), (r.zz_chain, s.zz_chain), (r.expect_x, s.expect_x),
                     (r.outcomes, s.outcomes)):
            assert x.tobytes() == y.tobytes(), (c["n"], c["precision"])
