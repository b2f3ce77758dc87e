"""CPU test of the heavy work lists' sizes (trident_amd/csrc/heavy_items.h):
tests/cpp/test_heavy_items.cpp is compiled with g++ and cuts rows of one to
nine column passes into windows and items over the whole tuning range."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_work_lists_hold_what_the_symbolic_cuts(tmp_path):
    exe = str(tmp_path / "test_heavy_items")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror",
                    os.path.join(ROOT, "tests", "cpp", "test_heavy_items.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "heavy items ok" in r.stdout
