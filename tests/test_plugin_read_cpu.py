"""The plugin reads a host scheduler's job through the public job API only (the
shortcut to a job's gates is the engine library's, for its own jobs)."""
import os
import subprocess
import sys

from conftest import ROOT

HOST = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
plug = ctypes.CDLL(sys.argv[2])
dumps = ctypes.c_int.in_dll(stub, "dumps")
class Options(ctypes.Structure):
    _fields_ = [(f, ctypes.c_int) for f in ("precision", "return_amplitudes", "return_probabilities", "return_expect_z",
                                            "fusion_max_qubits", "skip_shots", "blocked")]
out = (ctypes.c_char * 512)()
opts = Options(skip_shots=1)
plug.moonlab_mi355x_execute_ex.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
plug.moonlab_mi355x_execute_ex(8, ctypes.byref(opts), out)   # with a device or without: the job is read first
print(dumps.value)
"""


def test_plugin_reads_jobs_through_their_dump(tmp_path):
    stub = str(tmp_path / "job_stub.so")
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", os.path.join(ROOT, "tests", "job_stub.c"), "-o", stub], check=True)
    plugin = os.path.join(ROOT, "moonlab_amd", "lib", "libmoonlab_mi355x_plugin.so")
    r = subprocess.run([sys.executable, "-c", HOST, stub, plugin], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split()[-1] == "2"   # its size, then its text
