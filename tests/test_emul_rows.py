"""The 2D x-passes over blocks of neighbouring rows, built for the CPU with
AddressSanitizer (tests/emul), for plain and tangent-linear steps of many members:
in bounds, and equal to the FP64 oracle and to a single member's replay.  Takes some
minutes with the build, so it runs only with PSG_EMUL=1 in the environment."""
import os
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emul")


@pytest.mark.skipif(os.environ.get("PSG_EMUL") != "1", reason="host bounds-check build: set PSG_EMUL=1")
def test_emulated_rows_of_many_members():
    subprocess.check_call(["make", "-s", "-C", HERE, "-j8", "_build/rows_check"])
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1:detect_stack_use_after_return=0")
    r = subprocess.run([os.path.join(HERE, "_build", "rows_check")], env=env, capture_output=True, text=True, timeout=3000)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
