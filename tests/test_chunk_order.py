"""The order in which a launch's workgroups take chunks (csrc/chunks.hpp), compiled for the host against a model of
the device memory in which a request that nobody waits for arrives as late as it may: every launch hands out each
of its chunks exactly once and leaves the state for the next one, which would otherwise lose its first chunk and
wait for it forever."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_each_chunk_once_whatever_arrives_late(tmp_path):
    exe = str(tmp_path / "chunk_order")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "host", "chunk_order.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
