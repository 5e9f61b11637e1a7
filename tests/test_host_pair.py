"""The two parts of a mixed bitplane batch run on two host threads; what one of
them throws becomes its error code instead of the end of the process."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_exceptions_become_errors(tmp_path):
    exe = tmp_path / "host_pair_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-Werror", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "host_pair_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
