"""The packed search's device memory, under host emulation (tests/emu): a plan
whose allocations fail reports it on every such run and never launches with
part of its memory; it allocates what its launches can reach, and more when
the autotuner's settings ask for it."""
import os
import subprocess
import sys

import pytest

from test_emu import EMU, emu_lib  # noqa: F401


@pytest.mark.parametrize("case", ["pack out of memory", "pack memory", "pack grows"])
def test_packed_memory(emu_lib, case):  # noqa: F811
    env = dict(os.environ, RDMCE_LIB=emu_lib, EMU_CUS="1", EMU_BARRIER_TIMEOUT="120")
    r = subprocess.run([sys.executable, os.path.join(EMU, "run_cases.py"), case], capture_output=True, text=True,
                       timeout=600, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "ok" in r.stdout and "FAIL" not in r.stdout
