"""csrc/gemm_wide_rule.hpp on the host: the projections that the GPU tests of the wide-tile GEMM mean
to cover are the ones the rule sends there (256 compute units), and the row ranges of its comment."""
import os
import shutil
import subprocess

import pytest

import test_gpu_gemm_wide as W

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.fixture(scope="module")
def wins(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("rule") / "gemm_wide_rule")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "gemm_wide_rule.cpp")], check=True)

    def ask(shapes):
        args = [str(v) for s in shapes for v in s]
        out = subprocess.run([exe] + args, check=True, capture_output=True, text=True, timeout=60).stdout
        return [int(v) for v in out.split()]

    return ask


def test_covered_shapes(wins):
    for hidden, heads, ffn, vocab, rows, wide in W.CASES:
        shapes = {"qkv": ("int4", (heads + 2) * 128, hidden, rows), "wo": ("int4", hidden, hidden, rows),
                  "gate_up": ("int4", 2 * ffn, hidden, rows), "down": ("int4", hidden, ffn, rows),
                  "head": ("head", vocab, hidden, rows)}
        got = {n for n, w in zip(shapes, wins(shapes.values())) if w}
        assert got == set(wide), (hidden, rows, got)
    kw, rows = W.LATENT, W.LATENT_ROWS
    n = kw["n_heads"] * (kw["nope_dim"] + kw["rope_dim"]) + kw["latent_dim"] + kw["rope_dim"]
    assert wins([("int4", n, kw["hidden_dim"], rows)]) == [1]


@pytest.mark.parametrize("shape,ranges", [
    (("tuned", 22016, 4096), [(65, 128), (161, 256), (289, 513)]),
    (("tuned", 6144, 4096), [(225, 513)]),
    (("tuned", 4096, 11008), [(321, 513)]),
    (("tuned", 4096, 4096), [(353, 513)]),
    (("head", 32000, 4096), [(65, 128), (193, 256), (321, 384), (449, 512)])])
def test_row_ranges(wins, shape, ranges):
    got = wins([shape + (m,) for m in range(1, 514)])
    assert got == [int(any(a <= m <= b for a, b in ranges)) for m in range(1, 514)]
