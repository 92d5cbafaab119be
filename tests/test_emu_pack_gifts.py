"""Work handed to idle waves by the packed search, under host emulation
(tests/emu): half of a run's roots, every other record of the stack, and half
of one record's candidates, with clique lists, root statistics and batches.
The build looks for idle waves after every pass and counts the kinds of
gifts, so a case fails when its kind is never given."""
import os
import subprocess
import sys

import pytest

from test_emu import EMU, emu_lib  # noqa: F401


@pytest.mark.parametrize("case", ["pack gifts", "pack batch", "pack routed runs", "pack wide runs K90"])
def test_gifts_match_oracle(emu_lib, case):  # noqa: F811
    lib = os.path.join(EMU, "_build", "librdmce_emu_gifts.so")
    env = dict(os.environ, RDMCE_LIB=lib, EMU_CUS="1", EMU_BARRIER_TIMEOUT="120")
    r = subprocess.run([sys.executable, os.path.join(EMU, "run_cases.py"), case], capture_output=True, text=True,
                       timeout=600, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "ok" in r.stdout and "FAIL" not in r.stdout
