"""The sums of the diagonal elements on the CPU, with AddressSanitizer and
UndefinedBehaviorSanitizer: tests/native/diag_host.cpp."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_diagonal_sums(tmp_path):
    exe = str(tmp_path / "diag")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                           "-o", exe, os.path.join(HERE, "native", "diag_host.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
