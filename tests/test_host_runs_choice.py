"""The plain form's choice between runs and single kernels
(tests/cpp/runs_choice.cpp, on the CPU)."""
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
def test_runs_are_taken_where_they_are_faster(tmp_path):
    oracle_o, exe = str(tmp_path / "oracle.o"), str(tmp_path / "runs_choice")
    subprocess.check_call(["gcc", "-std=gnu11", "-O2", "-ffp-contract=off", "-fopenmp", "-c",
                           os.path.join(ROOT, "oracle", "qvnt_oracle.c"), "-o", oracle_o])
    subprocess.check_call([build.HIPCC, "-x", "c++", "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cpp", "runs_choice.cpp"),
                           os.path.join(ROOT, "qvnt_amd", "csrc", "runs.cpp"), "-x", "none", oracle_o, "-lgomp", "-lm", "-o", exe])
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
