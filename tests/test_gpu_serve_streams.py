"""A server runs on the streams it makes at its start, one per engine and large
worker, so that each has a hardware queue of its own: none is made later, for
co-batches of both precisions neither."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

HOST = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import moonlab_amd as m
made = ctypes.c_int.in_dll(stub, "streams_made")
srv = m.Server()
first = made.value
for _ in range(4):
    gates = [(4, q, -1, -1, 0.0) for q in range(8)]
    tickets = [srv.submit(8, gates, shots=4, seed=1, precision=k % 2) for k in range(40)]
    for t in tickets:
        assert srv.wait(t).status == 0
largest = srv.stats()["largest_batch"]
srv.close()
print(first, made.value, largest)
"""


def test_no_stream_is_made_after_the_start(tmp_path):
    stub = str(tmp_path / "alloc_limit.so")
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", os.path.join(ROOT, "tests", "alloc_limit.c"), "-o", stub, "-ldl"],
                   check=True)
    r = subprocess.run([sys.executable, "-c", HOST, stub, ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    first, made, largest = (int(x) for x in r.stdout.split()[-3:])
    assert first == made == 4 and largest > 1
