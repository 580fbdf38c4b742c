"""A tile's 16 loads are in flight together in every kernel that reads one:
from the compiler's own assembly, no wait for memory between them."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qvnt_amd"))
import build  # noqa: E402  (qvnt_amd/build.py: the library's own compile flags)

sys.path.pop(0)


def _runs_of_loads(body):
    """Lengths of the runs of global loads with neither a wait for vector memory nor a branch between them."""
    runs, n = [], 0
    for line in body.splitlines():
        op = line.strip()
        if op.startswith("global_load"):
            n += 1
        elif (op.startswith("s_waitcnt") and "vmcnt" in op) or op.startswith("s_cbranch"):
            runs.append(n)
            n = 0
    return runs


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_a_tiles_loads_do_not_wait_for_each_other(tmp_path):
    cmd = build.compile_command("fused.hip", str(tmp_path / "fused.o")) + ["--save-temps"]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600, cwd=str(tmp_path))
    assert res.returncode == 0, res.stderr
    asm = [p for p in os.listdir(tmp_path) if p.endswith(".s") and "gfx950" in p]
    assert len(asm) == 1, os.listdir(tmp_path)
    text = open(os.path.join(tmp_path, asm[0])).read()
    # (the persistent kernel holds the tile body twice: tiles of whole waves, and smaller ones)
    bodies = {"k_fusedId": 1, "k_fusedIf": 1, "k_batchId": 1, "k_batchIf": 1, "k_batch_persistId": 2, "k_batch_persistIf": 2}
    for kernel, copies in bodies.items():
        (name,) = re.findall(r"^(_ZN\S*\d%s\S*):" % kernel, text, re.M)
        body = text.split("\n%s:" % name, 1)[1].split(".Lfunc_end", 1)[0]
        assert sum(n >= 16 for n in _runs_of_loads(body)) >= copies, (kernel, sorted(_runs_of_loads(body))[-4:])


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_a_lanes_table_is_loaded_ahead(tmp_path):
    """The diagonal op whose table differs by lane: 16 phases in FP32, 8 and 8
    in FP64, asked for before the first is waited for."""
    cmd = build.compile_command("fused.hip", str(tmp_path / "fused.o")) + ["--save-temps"]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600, cwd=str(tmp_path))
    assert res.returncode == 0, res.stderr
    (asm,) = [p for p in os.listdir(tmp_path) if p.endswith(".s") and "gfx950" in p]
    text = open(os.path.join(tmp_path, asm)).read()
    # (beside the tile's own 16 loads)
    for kernel, ahead, groups in (("k_fusedId", 8, 2), ("k_fusedIf", 16, 1), ("k_batchId", 8, 2), ("k_batchIf", 16, 1)):
        (name,) = re.findall(r"^(_ZN\S*\d%s\S*):" % kernel, text, re.M)
        body = text.split("\n%s:" % name, 1)[1].split(".Lfunc_end", 1)[0]
        assert sum(n >= ahead for n in _runs_of_loads(body)) >= groups + 1, (kernel, sorted(_runs_of_loads(body))[-4:])
