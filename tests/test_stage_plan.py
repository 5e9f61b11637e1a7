"""A batch's results travel in pieces through a pinned ring of fixed size: the
division by itself."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_pieces_fit_the_ring(tmp_path):
    exe = tmp_path / "stage_plan_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "stage_plan_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
