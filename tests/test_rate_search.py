"""A decoded bitplane is returned only if every code its rate search tries below
the accepted one has run to its end: the rule by itself, on made-up records."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_unfinished_codes_are_found(tmp_path):
    exe = tmp_path / "rate_search_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "rate_search_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
