"""Host-only check of batches whose SpMV has more segments than a launch's block map
can name (one a problem and colour): 8191 and 8192 problems of eight colours, 936
and 937 of seventy, and the most problems a batch takes
(tests/cpp/batch_cut_test.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launches_hold_whole_problems(tmp_path):
    exe = str(tmp_path / "batch_cut_test")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O1", "--offload-arch=gfx950", "-x", "hip",
                        "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "batch_cut_test.cpp"),
                        "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    cases = {(1, 1): 1, (64, 8): 1, (8191, 8): 1, (8192, 8): 2, (936, 70): 1, (937, 70): 2, (65535, 1): 1,
             (65535, 8): 9, (2000, 128): 4, (511, 128): 1, (512, 128): 2}
    out = subprocess.run([exe], input="\n".join(f"{p} {s}" for p, s in cases) + "\n", capture_output=True, text=True,
                         timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split() == ["ok"] + [str(n) for n in cases.values()]
