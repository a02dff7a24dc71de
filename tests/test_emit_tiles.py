"""The tile emitter of csrc/uw_rows.h built for the host and run as workgroups of fibers (tests/cpp/host): compact
list, windows and their tails, halo cells, the plane-by-plane fallback of dense tiles, colours and collision
records, on grids of one row segment per row and of several, against a literal first-seen walk; and every tiling
that a launch can ask for."""
import os
import subprocess

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def test_emitter_on_the_host(tmp_path):
    exe = tmp_path / "emit_tiles"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wno-unknown-pragmas", "-Wno-unused-function",
                    "-I", os.path.join(CPP, "host"), "-o", str(exe), os.path.join(CPP, "emit_tiles.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", f"{r.returncode} {r.stdout[-2000:]} {r.stderr[-2000:]}"
