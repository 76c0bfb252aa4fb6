"""The server's block bookkeeping without a device: what its running jobs hold
and what it keeps for the next ones stay within its budget at every step of
random job mixes (C++ check of the header that the library uses)."""

import os
import shutil
import subprocess

import pytest


def test_kept_and_held_blocks_stay_within_the_budget(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    here = os.path.dirname(os.path.abspath(__file__))
    exe = str(tmp_path / "block_ledger_check")
    subprocess.run([gxx, "-std=c++17", "-O2", os.path.join(here, "cpp", "block_ledger_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    reused = [int(line.split()[-3]) for line in r.stdout.splitlines()]
    assert len(reused) == 3 and min(reused) > 100
