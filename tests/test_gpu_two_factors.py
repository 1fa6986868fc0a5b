"""tests/cpp/two_factors.cpp: a substitution uses the factorisation it is given, on meshes swept in LDS (where the
mesh holds the products of its last factorisation) and above."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "two_factors.bin")


@pytest.mark.parametrize("n", [2, 900, 20000, 20001])
def test_substitution_goes_with_its_factorisation(n):
    assert os.path.exists(EXE), "build the C++ callers first (__graft_entry__.build())"
    print("case: two factors", n, flush=True)
    r = subprocess.run([EXE, str(n)], capture_output=True, text=True, timeout=60)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok")
