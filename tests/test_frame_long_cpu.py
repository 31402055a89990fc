"""Planning a long circuit as rotation passes costs what its gates cost: 60
times the gates may take five times as long a gate, no more (a planner that
copied the pending gates at every phase and pass took 20 times as long)."""
import glob
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_planning_stays_linear(tmp_path):
    objs = sorted(glob.glob(os.path.join(ROOT, "moonlab_amd", "_build", "*.o")))
    if not objs or not os.path.exists(HIPCC):
        pytest.skip("engine objects not built (python -m moonlab_amd.build)")
    inc = ["-I" + os.path.join(ROOT, d) for d in ("include", "moonlab_amd/csrc")]
    exe = str(tmp_path / "frame_long")
    subprocess.run([HIPCC, "-O2", "-std=c++17", *inc, "-c", os.path.join(ROOT, "tests", "frame_long.cpp"),
                    "-o", str(tmp_path / "fl.o")], check=True, capture_output=True)
    subprocess.run([HIPCC, "--offload-arch=gfx950", str(tmp_path / "fl.o"), "-x", "none", *objs, "-o", exe, "-lpthread"],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    for line in r.stdout.splitlines():
        n, short, long = (float(x) for x in line.split())
        assert long < 5.0 * short, line
