"""NewHope's exact FP32 arithmetic mod q on the CPU: `make -C tests/c newhope-f32-run` builds
tests/c/newhope_f32_test.cpp with the host compiler (no floating-point contraction) and runs
it over pqc_amd/csrc/newhope_f32.h: products, reductions and the transforms' bounds."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_newhope_f32_arith_mod_q():
    r = subprocess.run(["make", "-C", os.path.join(ROOT, "tests", "c"), "newhope-f32-run"], capture_output=True,
                       text=True, timeout=300)
    out = r.stdout + r.stderr
    assert r.returncode == 0, out[-4000:]
    assert "NewHope f32 arithmetic mod q: all checks hold" in out
