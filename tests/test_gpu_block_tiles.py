"""Fused circuits whose blocks share passes over 12-qubit tiles: one tile and
a few more, every block width, lone gates among the blocks, blocks on the
highest and on scattered qubits."""
import numpy as np
import pytest

from conftest import random_gate_list, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [11, 12, 13, 16])
@pytest.mark.parametrize("kmax", [1, 2, 3, 4, 5])
def test_fused_vs_oracle(eng, oracle, n, kmax):
    from moonlab_amd import workloads
    rng = np.random.default_rng(10 * n + kmax)
    a0 = random_state(n, rng)
    neighbours = workloads.su2_cz_circuit(n, 3, n)
    neighbours = [tuple(r) for r in neighbours.tolist()]
    for gates in (neighbours, random_gate_list(n, 40, rng), [(4, n - 1, -1, -1, 0.0)]):
        want = oracle.apply(n, a0.copy(), gates)
        for prec, tol in ((eng.C128, 1e-12), (eng.C64, 2e-5)):
            with eng.StateVector(n, prec) as sv:
                got = sv.load(a0).apply(gates, fuse=kmax).amplitudes()
            assert np.max(np.abs(got - want)) < tol, (n, kmax, prec, len(gates))
