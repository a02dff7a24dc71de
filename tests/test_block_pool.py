"""The pool of kept device blocks (csrc/uw_blocks.h), built for the host: bounds on its size and on the slack
of a block it hands out, oldest blocks let go first, every block with one owner."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_block_pool(tmp_path):
    exe = tmp_path / "block_pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), os.path.join(HERE, "cpp", "block_pool.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
