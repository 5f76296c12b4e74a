"""The LDS room of an operator's terms on the CPU: tests/native/lds_plan_host.cpp."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_lds_plan(tmp_path):
    exe = str(tmp_path / "lds_plan")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                           "-o", exe, os.path.join(HERE, "native", "lds_plan_host.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
