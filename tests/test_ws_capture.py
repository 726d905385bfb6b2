"""The workspace registry (ws_registry.h) under stream capture, on the CPU: a
recorded call's new buffer is taken apart from the captured stream and zeroed at
once, nothing is freed on that stream, and a buffer that a graph may use keeps
its address until its stream is released, with a bound on what is kept."""
import os
import subprocess
import tempfile

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_recorded_calls_allocate_nothing_on_the_captured_stream():
    src = os.path.join(REPO, "tests", "ws_capture_check.cpp")
    inc = os.path.join(REPO, "sneppx-alg_amd", "csrc")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "ws_capture")
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", inc, src, "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        assert "ok:" in r.stdout
