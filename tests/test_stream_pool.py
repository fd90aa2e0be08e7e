"""Workspaces by stream, on the CPU: tests/cpp/stream_pool_check.cpp, built by
the package Makefile."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(REPO, "tests", "cpp", "bin", "stream_pool_check")


def test_stream_pool():
    if not os.path.exists(BIN):
        subprocess.run(["make", "-C", os.path.join(REPO, "mlx-confucius4-tts_amd"),
                        "../tests/cpp/bin/stream_pool_check"], check=True)
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout == "0 failures\n"
