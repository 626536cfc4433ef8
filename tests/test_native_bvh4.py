"""Native CPU test of the 4-wide quantised BVH builder (tests/native/test_bvh4.cpp)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent


def test_bvh4_structure_native(tmp_path):
    exe = tmp_path / "test_bvh4"
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", str(ROOT / "native" / "test_bvh4.cpp"),
                    str(ROOT.parent / "merian_amd" / "csrc" / "bvh.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
