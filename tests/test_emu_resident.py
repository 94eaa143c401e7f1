"""The resident kernels' transforms on the CPU (tests/emu/line_emu.cpp): values,
LDS slots in range, and no two threads on one slot without a barrier between."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("checks", ["address,undefined", "thread"])
def test_line_transforms_under_sanitizers(tmp_path, checks):
    exe = str(tmp_path / "line_emu")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wno-unknown-pragmas", f"-fsanitize={checks}",
                    "-fno-sanitize-recover=all", "-I",
                    os.path.join(ROOT, "als_speckle_amd", "csrc"),
                    os.path.join(ROOT, "tests", "emu", "line_emu.cpp"), "-o", exe, "-pthread"],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and "0 bad" in r.stdout, r.stdout[-2000:] + r.stderr[-4000:]
