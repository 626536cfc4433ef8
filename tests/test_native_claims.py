"""Native CPU test of the division of rays among work cursors (tests/native/test_ray_claims.cpp)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent


def test_ray_claims_native(tmp_path):
    exe = tmp_path / "test_ray_claims"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", str(ROOT / "native" / "test_ray_claims.cpp"), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
