"""The host rules of a launch (workgroups, chunks, which launches claim and whose
counters they take), checked on the CPU by the compiled program
tests/hip/launch_rules."""
import subprocess
from pathlib import Path

import pytest

PROG = Path(__file__).resolve().parent / "hip" / "launch_rules"


def test_launch_rules():
    if not PROG.exists():
        pytest.fail(f"{PROG} is not built (run __graft_entry__.build())")
    res = subprocess.run([str(PROG)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
