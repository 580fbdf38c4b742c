"""Register allocation of the run kernels (runs.hip), from the compiler's own
resource report: the 8 or 16 amplitudes a thread holds stay in VGPRs, in all
four variants, with four waves a SIMD."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qvnt_amd"))
import build  # noqa: E402  (qvnt_amd/build.py: the library's own compile flags)

sys.path.pop(0)


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_run_kernels_do_not_spill(tmp_path):
    cmd = build.compile_command("runs.hip", str(tmp_path / "runs.o")) + ["-Rpass-analysis=kernel-resource-usage"]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr
    kernels = {}
    for block in res.stderr.split("Function Name: ")[1:]:
        name = block.split()[0]
        if "k_run" in name:
            kernels[name] = {k: int(re.search(re.escape(k) + r": (\d+)", block)[1])
                             for k in ("ScratchSize [bytes/lane]", "VGPRs Spill", "SGPRs Spill", "Occupancy [waves/SIMD]")}
    assert len(kernels) == 4, res.stderr
    for name, k in kernels.items():
        assert k == {"ScratchSize [bytes/lane]": 0, "VGPRs Spill": 0, "SGPRs Spill": 0, "Occupancy [waves/SIMD]": 4}, (name, k)
