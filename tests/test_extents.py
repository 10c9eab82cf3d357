"""Index arithmetic of the stage kernels at the largest accepted problem
(n = 2048): a tile of panel 6 against the same tile of panel 1, whose byte
offsets are small, in full-size sparse arrays (tests/emu/extent_check.cpp)."""
import os
import subprocess


def test_offsets_at_the_largest_problem(tmp_path):
    here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
    exe = str(tmp_path / "extent_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", f"-I{here}", "-o", exe,
                    os.path.join(here, "extent_check.cpp")], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-3000:] + p.stderr[-1000:]
