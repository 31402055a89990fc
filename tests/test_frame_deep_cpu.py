"""Deep circuits of the Pauli-rotation engine on the host (no device):
tests/frame_deep.cpp runs passes of up to 8000 rotations thread by thread
against the oracle, both precisions, last passes and earlier ones."""
import glob
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_frame_programs_of_deep_circuits(tmp_path):
    objs = sorted(glob.glob(os.path.join(ROOT, "moonlab_amd", "_build", "*.o")))
    if not objs or not os.path.exists(HIPCC):
        pytest.skip("engine objects not built (python -m moonlab_amd.build)")
    inc = ["-I" + os.path.join(ROOT, d) for d in ("include", "moonlab_amd/csrc", "oracle", "tests")]
    exe = str(tmp_path / "frame_deep")
    subprocess.run(["gcc", "-O2", "-march=x86-64-v3", "-fopenmp", "-c", os.path.join(ROOT, "oracle", "sv_oracle.c"),
                    "-I" + os.path.join(ROOT, "oracle"), "-o", str(tmp_path / "svo.o")], check=True)
    subprocess.run([HIPCC, "-O2", "-std=c++17", *inc, "-c", os.path.join(ROOT, "tests", "frame_deep.cpp"),
                    "-o", str(tmp_path / "fd.o")], check=True, capture_output=True)
    subprocess.run([HIPCC, "--offload-arch=gfx950", str(tmp_path / "fd.o"), str(tmp_path / "svo.o"), "-x", "none",
                    *objs, "-o", exe, "-lpthread", "-fopenmp"], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok:"), r.stdout
