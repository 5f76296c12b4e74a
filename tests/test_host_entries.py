"""Host-side tables of the products on the CPU: the parity entries against
term-by-term matching (tests/native/entries_host.cpp) and the window
canonicaliser against brute force (tests/native/window_host.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("name", ["entries", "window"])
def test_native(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "native", f"{name}_host.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
