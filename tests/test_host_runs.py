"""The plain form's runs (qvnt_amd/csrc/runs.cpp, runs_ops.hpp) on the CPU:
tests/cpp/runs_model.cpp plans random circuits of every gate kind, runs the
kernel's own gate code tile by tile and compares every run's state with the
oracle's, bit for bit, in both precisions."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qvnt_amd"))
import build  # noqa: E402  (qvnt_amd/build.py: the compiler's path)

sys.path.pop(0)


@pytest.mark.skipif(not os.path.exists(build.HIPCC) or shutil.which("gcc") is None, reason="needs hipcc and gcc")
def test_runs_equal_the_oracle_bit_for_bit(tmp_path):
    oracle_o, exe = str(tmp_path / "oracle.o"), str(tmp_path / "runs_model")
    subprocess.check_call(["gcc", "-std=gnu11", "-O2", "-ffp-contract=off", "-fopenmp", "-c",
                           os.path.join(ROOT, "oracle", "qvnt_oracle.c"), "-o", oracle_o])
    # only the host side is compiled: the same formulas, rounded the same way
    objects = []
    for src in (os.path.join(ROOT, "tests", "cpp", "runs_model.cpp"), os.path.join(ROOT, "qvnt_amd", "csrc", "runs.cpp")):
        obj = str(tmp_path / (os.path.basename(src) + ".o"))
        subprocess.check_call([build.HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=" + build.ARCH, "-std=c++17", "-O1",
                               "-ffp-contract=off", "-c", src, "-o", obj])
        objects.append(obj)
    subprocess.check_call([build.HIPCC, *objects, oracle_o, "-lgomp", "-lm", "-o", exe])
    res = subprocess.run([exe], capture_output=True, text=True, timeout=600, env=dict(os.environ, OMP_NUM_THREADS="1"))
    print(res.stdout)
    assert res.returncode == 0, res.stdout + res.stderr
    assert "equal to the oracle" in res.stdout
