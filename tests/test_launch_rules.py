"""The rules that choose between launches, against measured times of both sides (tests/host/launch_rules.cpp; the rules are the library's own headers)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rules_take_the_faster_side(tmp_path):
    exe = str(tmp_path / "launch_rules")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "host", "launch_rules.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
