"""A pinned host block that ends while the host is out of memory
(tests/cpp/host_block.cpp, on the CPU with its own allocators)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qvnt_amd"))
import build  # noqa: E402  (qvnt_amd/build.py: the compiler's path)

sys.path.pop(0)


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_a_block_ends_without_memory(tmp_path):
    exe = str(tmp_path / "host_block")
    subprocess.check_call([build.HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=" + build.ARCH, "-std=c++17", "-O1",
                           os.path.join(ROOT, "tests", "cpp", "host_block.cpp"), "-x", "none", build.LIB_PATH,
                           "-Wl,-rpath," + build.LIB_DIR, "-o", exe])
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
