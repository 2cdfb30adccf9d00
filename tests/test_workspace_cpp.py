"""Runs tests/cpp/test_workspace.cpp: the bookkeeping of the library-owned scratch
on the CPU, two host threads on one stream among its cases."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
BIN = os.path.join(HERE, "cpp", "_build", "test_workspace")


def test_workspace_bookkeeping():
    if not os.path.exists(BIN):   # normally built by __graft_entry__.build()
        subprocess.run(["make", "-s", "-C", os.path.join(HERE, "cpp"), "_build/test_workspace"], check=True)
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "0 failure(s)" in r.stdout
