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


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel by kernel, the assembly of fused.hip."""
    if not os.path.exists(build.HIPCC):
        pytest.skip("needs hipcc")
    tmp = tmp_path_factory.mktemp("asm")
    cmd = build.compile_command("fused.hip", str(tmp / "fused.o")) + ["--save-temps"]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600, cwd=str(tmp))
    assert res.returncode == 0, res.stderr
    (asm,) = [p for p in os.listdir(tmp) if p.endswith(".s") and "gfx950" in p]
    text = open(os.path.join(tmp, asm)).read()
    out = {}
    for kernel in ("k_fusedId", "k_fusedIf", "k_batchId", "k_batchIf", "k_batch_persistId", "k_batch_persistIf"):
        (name,) = re.findall(r"^(_ZN\S*\d%s\S*):" % kernel, text, re.M)
        out[kernel] = text.split("\n%s:" % name, 1)[1].split(".Lfunc_end", 1)[0]
    return out


def test_a_tiles_loads_do_not_wait_for_each_other(kernels):
    for kernel, body in kernels.items():
        # (the persistent kernel holds the tile body twice: tiles of whole waves, and smaller ones)
        copies = 2 if "persist" in kernel else 1
        assert sum(n >= 16 for n in _runs_of_loads(body)) >= copies, (kernel, sorted(_runs_of_loads(body))[-4:])


def test_a_lanes_table_is_loaded_ahead(kernels):
    """The diagonal op whose table differs by lane: 16 phases in FP32, 8 and 8
    in FP64, asked for before the first is waited for (beside the tile's own 16 loads)."""
    for kernel, ahead, groups in (("k_fusedId", 8, 2), ("k_fusedIf", 16, 1), ("k_batchId", 8, 2), ("k_batchIf", 16, 1)):
        runs = _runs_of_loads(kernels[kernel])
        assert sum(n >= ahead for n in runs) >= groups + 1, (kernel, sorted(runs)[-4:])
