"""Device and pinned memory of the engine library, counted allocation by
allocation on the CPU emulation of the kernels (tests/emu): estimates and
budgets against what is allocated, and calls that are to work where memory for
their faster form is missing.  Each check of tests/emu/limits_driver.py
runs in a process of its own, since it loads the emulated library."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "emu"))

import build_emu  # noqa: E402


@pytest.mark.parametrize("check", ["estimate", "server", "costs", "images", "paths", "long_paths"])
def test_emulated_limits(check):
    lib = build_emu.build()
    env = dict(os.environ)
    env["LD_LIBRARY_PATH"] = os.path.dirname(lib) + (
        ":" + env["LD_LIBRARY_PATH"] if env.get("LD_LIBRARY_PATH") else "")
    env.update(EMU_CUS="3", EMU_OCC="2")
    p = subprocess.run([sys.executable, os.path.join(HERE, "emu", "limits_driver.py"), lib, check],
                       capture_output=True, text=True, timeout=600, env=env)
    assert p.returncode == 0, p.stdout + p.stderr
    assert json.loads(p.stdout.strip().splitlines()[-1])["failures"] == [], p.stdout
