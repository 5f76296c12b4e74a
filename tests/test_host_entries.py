"""The products' parity entries against term-by-term matching, on the CPU
(tests/native/entries_host.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_entries_match_as_their_terms(tmp_path):
    exe = str(tmp_path / "entries")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "native", "entries_host.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
