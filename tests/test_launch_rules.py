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


def test_smallest_pool(tmp_path):
    """Robots by their bodies, piles by how many copies of a body's ground contact their list holds:
    (free bodies, list, most valid slots seen settled) in the extended mode, never below the last
    number with the list's own length as the bound; (free, round, list, valid slots of 99 in a hundred
    environments) in the reference's mode."""
    extended = [(12, 64, 22), (12, 128, 21), (24, 64, 59), (24, 80, 58), (24, 128, 33), (24, 200, 24), (38, 64, 62), (38, 80, 76),
                (38, 128, 90), (38, 200, 56), (38, 256, 35), (50, 128, 100), (50, 200, 96), (50, 256, 68), (50, 384, 26),
                (62, 128, 108), (62, 200, 115), (62, 256, 120), (62, 384, 69), (62, 512, 30)]
    plain = [(12, 8, 64, 12), (24, 16, 64, 36), (40, 27, 64, 40), (50, 34, 64, 37), (64, 43, 64, 43), (64, 43, 128, 71), (40, 27, 200, 36)]
    rows = run(tmp_path, "\n".join([f'printf("%u\\n", pool_floor(0, {n}, {n}, {m}, true));' for n, m, _ in extended]
                                   + [f'printf("%u\\n", pool_floor(0, {n}, {r}, {m}, false));' for n, r, m, _ in plain])
               + 'for (bool e : {false, true}) printf("%u %u %u %u\\n", pool_floor(13, 0, 0, 64, e), pool_floor(29, 0, 0, 64, e),'
                 ' pool_floor(1, 0, 0, 1, e), pool_floor(13, 2, 2, 64, e));')
    for (n, m, most), (slots,) in zip(extended, rows):
        assert min(slots, m) >= most, (n, m, slots, most)
    for (n, r, m, most), (slots,) in zip(plain, rows[len(extended):]):
        assert min(slots, m) >= most, (n, r, m, slots, most)
    assert rows[-2:] == [[24, 32, 24, 24]] * 2


def test_steps_of_a_captured_launch(tmp_path):
    """Up to 64 substeps or one step, what is left of the schedule, and no product past 32 bits."""
    cases = [(1, 130), (1, 3), (2, 130), (5, 130), (63, 9), (64, 9), (65, 9), (1 << 26, 64), (0xFFFFFFFF, 64), (0, 70)]
    rows = run(tmp_path, "\n".join(f'printf("%u\\n", fused_calls({s}u, {left}u));' for s, left in cases))
    assert [n for n, in rows] == [64, 3, 32, 12, 1, 1, 1, 1, 1, 64]
    assert all(n * s < 1 << 32 for (n,), (s, _) in zip(rows, cases))


def test_every_joint_record_has_both_headers(tmp_path):
    """The lanes of a pair form their addresses from the half records' headers before the type is
    told apart: bodies, multiplier and type stand in both halves, whatever the type, and the second
    anchor keeps out of them."""
    rows = run(tmp_path, """
    const uint32_t types[] = {C_POSITIONAL, C_WELD, C_ANGULAR, C_ANGULAR_LIMIT, C_LINEAR_LIMIT, C_SLIDER};
    std::vector<ConstraintRec> t(6);
    std::vector<uint32_t> ranges;
    for (uint32_t k = 0; k < 6; ++k) {
        t[k] = ConstraintRec{};
        t[k].indices[0] = 2 * k + 1; t[k].indices[1] = 2 * k + 2; t[k].indices[3] = types[k];
        t[k].anchor_b[0] = 0.25f; t[k].anchor_b[1] = 100.0f; t[k].anchor_b[2] = -3.0f;
        t[k].limits[0] = -0.1f; t[k].limits[1] = 0.1f;
        ranges.push_back(k); ranges.push_back(1);
    }
    std::vector<float> im(4 * 13, 1.0f), com(4 * 13, 0.0f);
    std::vector<float4> q;
    std::vector<JointPhase> ph;
    build_joint_program(t, ranges, im.data(), com.data(), q, ph);
    auto u = [](float f) { uint32_t x; std::memcpy(&x, &f, 4); return x; };
    for (size_t r = 0; r + kJRecQuads <= q.size(); r += kJRecQuads)
        for (size_t h : {0, 4}) printf("%u %u %u %u\\n", u(q[r + h].x), u(q[r + h].y), u(q[r + h].z), u(q[r + h].w) >> 8);
""")
    assert rows == [[2 * k + 1, 2 * k + 2, k, t] for k, t in enumerate([2, 7, 3, 4, 5, 10]) for _ in range(2)]
