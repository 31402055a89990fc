"""Blocks of one and two qubits and lone gates that share a pass over 12-qubit
tiles: an amplitude that is not a number reaches no amplitude that the gates
themselves do not take it to, and the others are the oracle's."""
import numpy as np
import pytest

from conftest import random_gate_list, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12, 14])
def test_nan_stays_where_the_gates_take_it(eng, oracle, n):
    rng = np.random.default_rng(n)
    lone = [(12, 5, 0), (10, 1, 6), (16, 2, -1, -1, 0.7), (4, 3), (13, 4, 7), (23, 8, 9, 10), (19, 11, 2, -1, 0.4),
            (18, n - 1, 0, -1, 1.1), (24, 6, 5, 4), (2, 9), (17, 8, -1, -1, 0.3, 0.2, 0.1)]
    for gates in (lone, random_gate_list(n, 30, rng)):
        a = random_state(n, rng)
        a[rng.integers(0, 1 << n, size=5)] = complex(np.nan, np.nan)
        want = oracle.apply(n, a.copy(), gates)
        nan = np.isnan(want)
        assert nan.any() and not nan.all()
        for prec, tol in ((eng.C128, 1e-12), (eng.C64, 2e-5)):
            with eng.StateVector(n, prec) as sv:
                got = sv.load(a).apply(gates, fuse=1).amplitudes()
            assert not (np.isnan(got) & ~nan).any(), prec
            assert np.max(np.abs(got[~nan] - want[~nan])) < tol, prec


@pytest.mark.parametrize("n", [12, 13, 16])
def test_small_blocks_vs_oracle(eng, oracle, n):
    rng = np.random.default_rng(n)
    for kmax in (1, 2, 3):
        a = random_state(n, rng)
        gates = random_gate_list(n, 60, rng)
        want = oracle.apply(n, a.copy(), gates)
        for prec, tol in ((eng.C128, 1e-12), (eng.C64, 2e-5)):
            with eng.StateVector(n, prec) as sv:
                got = sv.load(a).apply(gates, fuse=kmax).amplitudes()
            assert np.max(np.abs(got - want)) < tol, (kmax, prec)
