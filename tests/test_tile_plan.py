"""CPU check of the W4A16 tile GEMM's plan (tile shape and K split): builds
tests/cpp/tile_plan_check.hip (host code only) and runs it."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_tile_plans(tmp_path):
    exe = tmp_path / "tile_plan_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-x", "c++", str(ROOT / "tests" / "cpp" / "tile_plan_check.hip"), "-o",
                    str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
