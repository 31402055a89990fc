"""Calls whose optional device memory cannot be had run without it and give
the same results.  The allocations are refused on the host, by
tests/alloc_limit.c in a process of its own."""
import json
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

HOST = """
import ctypes, json, sys
import numpy as np
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import moonlab_amd as m
limit, refused = ctypes.c_size_t.in_dll(stub, "alloc_limit_bytes"), ctypes.c_int.in_dll(stub, "alloc_refused")
def limited(nbytes, call):
    first = call()
    limit.value, refused.value = nbytes, 0
    second = call()
    limit.value = 2 ** 64 - 1
    return {"first": first, "second": second, "refused": refused.value}
"""


def run(tmp_path, code, refused=True):
    stub = str(tmp_path / "alloc_limit.so")
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", os.path.join(ROOT, "tests", "alloc_limit.c"), "-o", stub, "-ldl"],
                   check=True)
    r = subprocess.run([sys.executable, "-c", HOST + code, stub, ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert (out["refused"] > 0) == refused
    return out


@pytest.mark.parametrize("prec", [0, 1])
def test_shots_without_the_cumulative_table(tmp_path, prec):
    out = run(tmp_path, f"""
rng = np.random.default_rng(5)
sv = m.StateVector(16, {prec})
a = rng.normal(size=1 << 16) + 1j * rng.normal(size=1 << 16)
sv.load(a / np.linalg.norm(a))
u = rng.uniform(size=8 * 16 + 40)
print(json.dumps(limited(8 << 16, lambda: np.asarray(sv.sample(u)).tolist())))
""")
    assert out["first"] == out["second"]


def test_batch_without_slots_of_its_circuits_own(tmp_path):
    out = run(tmp_path, """
rng = np.random.default_rng(6)
terms = [(1.0, "".join("IXYZ"[k] for k in rng.integers(0, 4, size=12))) for _ in range(100)]
def circuit(k):
    gates = [(8, q, -1, -1, float(rng.uniform(0, 6))) for q in range(12)] + [(10, q + 1, q) for q in range(11)]
    return {"n": 12, "gates": gates, "precision": k % 2, "pauli": terms}
circuits = [circuit(k) for k in range(16)]
b = m.Batch()
def call():
    global b
    b.free()
    b = m.Batch()
    return [(r.norm, r.expect_z.tolist(), r.pauli_expect.tolist()) for r in b.run(circuits)]
print(json.dumps(limited(1 << 20, call)))
""")
    assert out["first"] == out["second"]


def test_batch_scratch_of_both_precisions_in_one_budget(tmp_path):
    # 140 circuits of 24 qubits: slots of 256 MiB, 16 GiB of them (a quarter more is asked for) for both precisions
    out = run(tmp_path, """
b = m.Batch()
limit.value = (20 << 30) + (1 << 20)
r = b.run([{"n": 24, "gates": [], "precision": k % 2} for k in range(140)])
print(json.dumps({"refused": refused.value, "ok": all(x.norm == 1.0 and np.all(x.expect_z == 1.0) for x in r)}))
""", refused=False)
    assert out["ok"]


def test_jobs_without_memory_for_their_program(tmp_path):
    out = run(tmp_path, """
rng = np.random.default_rng(7)
job = m.Job(13)
for _ in range(6):
    for q in range(13):
        job.add_gate(8, q, -1, float(rng.uniform(0, 6)))
    for q in range(12):
        job.add_gate(10, q + 1, q)
def call():
    r = job.execute_ex(amplitudes=True, expect_z=True, skip_shots=True)
    return r.amplitudes.view(np.float64).tolist() + r.expect_z.tolist()
r = limited(1, call)
print(json.dumps({"refused": r["refused"], "worst": max(abs(a - b) for a, b in zip(r["first"], r["second"]))}))
""")
    assert out["worst"] < 1e-12


def test_small_blocks_without_memory_for_their_steps(tmp_path):
    out = run(tmp_path, """
from moonlab_amd import workloads
sv, g = m.StateVector(14), workloads.su2_cz_circuit(14, 3, 1)
r = limited(1, lambda: sv.reset().apply(g, fuse=2).amplitudes().view(np.float64).tolist())
print(json.dumps({"refused": r["refused"], "worst": max(abs(a - b) for a, b in zip(r["first"], r["second"]))}))
""")
    assert out["worst"] < 1e-12
