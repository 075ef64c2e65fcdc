"""CPU check of the FP64 recursion engine: the host tables of
public_amd/csrc/line_rec.hpp, applied by a CPU emulation of the device's
steps, reproduce the oracle's LU-based derivative and filter cores to
rounding, for every scheme, periodic and open (padded) lines, lines of fewer
blocks than the window, and filter parameters up to the engine's limit
(beyond it the filter keeps the cyclic reduction)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_recursion_engine_matches_lu_cores(tmp_path):
    exe, obj = tmp_path / "line_rec_check", tmp_path / "oracle.o"
    src = os.path.join(ROOT, "tests", "cpp", "line_rec_check.cpp")
    orc = os.path.join(ROOT, "oracle", "cruna_oracle.c")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-c", orc, "-o", str(obj)], check=True)
    subprocess.run(["g++", "-O2", "-std=c++17", src, str(obj), "-o", str(exe), "-lm"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    rows = [line.split() for line in out.strip().splitlines()]
    assert len(rows) == 4 * 8 + 5 * 20 + 9 * 4 + 10 * 4
    for kind, scheme, n, alpha, usable, err in rows:
        assert int(usable) == (kind != "filter" or abs(float(alpha)) < 0.4972), (kind, alpha)
        # a filter's B has the condition number 1 / (1 - 2 |alpha|)
        tol = 1e-14 * max(1.0, 0.1 / (1.0 - 2.0 * min(abs(float(alpha)), 0.4972))) if kind == "filter" else 1e-14
        assert float(err) < tol, (kind, scheme, n, alpha, err)
