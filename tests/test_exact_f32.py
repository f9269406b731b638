"""csrc/exact_f32.hpp on the host: the branch-free exponentials and quotients that the exact sums
of the acceptance kernel are built from (softmax and renormalisation, sampler.rs:280-347) equal
(float)exp((double)x) and x / d over all magnitudes, subnormal results (low temperatures) and ties
among them, but for the rare exponentials that they leave to the plain form."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_branch_free_forms(tmp_path):
    exe = str(tmp_path / "exact_f32")
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "exact_f32.cpp")], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=300).stdout
    rows = {n: tuple(map(int, v)) for n, *v in map(str.split, out.splitlines())}
    assert set(rows) == {"exp_negative", "exp_subnormal", "exp_positive", "div_any", "div_low", "div_tie", "div_special"}
    for name, (n, wrong, _) in rows.items():
        assert n > 100 and wrong == 0, (name, n, wrong)
    # share of the exponentials left to the plain form: a bracket of 2^-41 in a spacing of at least 2^-24
    for name in ("exp_negative", "exp_subnormal", "exp_positive"):
        n, _, bad = rows[name]
        assert bad < n * 2.0 ** -16, (name, n, bad)
