"""Host-side logic and tables on the CPU, built with AddressSanitizer and
UndefinedBehaviorSanitizer: the programs of tests/native say what each compares."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("name", ["diag", "images", "grid", "lds_plan", "entries", "window"])
def test_native(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                           "-o", exe, os.path.join(HERE, "native", f"{name}_host.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
