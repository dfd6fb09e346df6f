"""The planner of the GEMM calls (csrc/q4_gemm_plan.h) on the host, by tests/c/gemm_plan.cpp: its closed
form for one weight and its levels for several give what handing out every workgroup gives; a weight alone
takes the shape and K split that are estimated to be its fastest, stores one by one among what they take (held
back for calls of several only where the weight fills more than half of the chip without a split and has a
short chain), and up to 128 rows the kernel that was timed faster for it; the
weights of an fp32 call of more rows take one kernel together, for no more time than the others' one launch; an order of blocks that is asked for
gives every weight its own launch; and a call's plan takes a fraction of its smallest kernel (0.4 to 0.9 us on
one core; a simulated schedule for every K split of every weight took 3.5 to 7.9)."""
import os
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_gemm_plans():
    program = os.fspath(HERE / "c" / "build" / "gemm_plan")
    subprocess.run(["make", "-C", os.fspath(HERE / "c"), program], check=True, capture_output=True)
    done = subprocess.run([program], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout
    *checks, a, b, c, d = done.stdout.splitlines()
    assert checks == ["schedule ok", "choices ok", "widths ok", "rows ok", "pairs ok", "order ok"]
    # between what they take (0.9, 0.8, 0.5, 0.4) and what that schedule took (7.9, 7.2, 4.8, 3.5), for a slower host's sake
    for line, most in zip((a, b, c, d), (5.0, 4.5, 3.0, 2.2)):
        name, us = line.split()
        assert float(us) < most, line
