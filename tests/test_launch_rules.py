"""The host's launch rules (zeno_amd/csrc/step.h), compiled on their own for the CPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "zeno_amd" / "csrc"
ROCM = Path("/opt/rocm/include")
CXX = shutil.which("g++")

pytestmark = pytest.mark.skipif(CXX is None or not (ROCM / "hip" / "hip_runtime.h").exists(), reason="needs g++ and the HIP headers")


def run(tmp_path, body: str):
    src = tmp_path / "rules.cpp"
    src.write_text('#include <cstdio>\n#include "step.h"\nusing namespace za;\nint main() {\n' + body + "\n}\n")
    exe = tmp_path / "rules"
    subprocess.run([CXX, "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return [[int(x) for x in line.split()] for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]


def test_workgroups_that_the_lds_holds(tmp_path):
    """Whole units of 1280 bytes; the largest sizes of which n fit, and the next."""
    rows = run(tmp_path, 'for (size_t b : {53760, 53761, 81920, 81921, 12800, 12801, 163840, 163841, 1, 0})'
                         ' printf("%zu %zu\\n", b, lds_workgroups(b));')
    assert dict(rows) == {53760: 3, 53761: 2, 81920: 2, 81921: 1, 12800: 12, 12801: 11, 163840: 1, 163841: 0, 1: 128, 0: 163840}
