"""How the threads of a compiled graph's attention launch share the copies in front of it, walked on the CPU up to the largest launch there is
(tests/host/graph_shares.cpp; the arithmetic is the kernel's own header)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copied_rows_are_shared_without_a_gap_and_nothing_is_stored_past_them(tmp_path):
    exe = str(tmp_path / "graph_shares")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "host", "graph_shares.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:]
