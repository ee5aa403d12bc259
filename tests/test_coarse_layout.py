"""Host-only check of a coarse plan's allocation: its parts start where their types
may, for even and odd counts of steps (a bottom level of eight colours has 15) and
one to four levels (tests/cpp/coarse_layout_test.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_parts_are_aligned(tmp_path):
    exe = str(tmp_path / "coarse_layout_test")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O1", "--offload-arch=gfx950", "-x", "hip",
                        "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "coarse_layout_test.cpp"),
                        "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lines = [f"{rows} {steps} {levels}" for rows in (1, 64, 585, 4681) for steps in (1, 2, 15, 45, 46, 135)
             for levels in (1, 2, 4)]
    out = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split() == ["ok", str(len(lines))]
