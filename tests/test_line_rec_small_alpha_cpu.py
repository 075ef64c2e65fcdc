"""FP64 filters of small alpha: the recursions' root keeps its digits however
small alpha is, and no alpha that the filter's LU core takes is refused."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_small_alphas_match_lu_core(tmp_path):
    exe, obj = tmp_path / "line_rec_small_check", tmp_path / "oracle.o"
    src = os.path.join(ROOT, "tests", "cpp", "line_rec_small_check.cpp")
    orc = os.path.join(ROOT, "oracle", "cruna_oracle.c")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-c", orc, "-o", str(obj)], check=True)
    subprocess.run(["g++", "-O2", "-std=c++17", src, str(obj), "-o", str(exe), "-lm"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    rows = [line.split() for line in out.strip().splitlines()]
    assert len(rows) == 15 * 2 * 8
    for scheme, n, alpha, usable, err in rows:
        assert usable == "1" and err != "refused", (scheme, n, alpha)
        # B is the identity to within alpha: the engine's general tolerance
        assert float(err) < 1e-14, (scheme, n, alpha, err)
