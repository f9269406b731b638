"""Projections whose row and column blocks fill the part run in the wide-tile GEMM: parity of
the whole forward with the oracle (QatLinear::forward, quant/src/qat.rs:315-348) at the edges of
its 64-row blocks, with a partial row chunk, a partial last column block and an odd number of
128-column groups (the two K-waves then take different counts).
Bar: logits and hidden states within 2e-3 relative per row, as for every quantised forward."""
import numpy as np
import pytest

import aarambh_hip as A
import refcpu as R
from gpu_util import make_pair, rel_rows

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.mark.parametrize("hidden,heads,ffn,vocab,rows", [
    (1920, 15, 12160, 1024, 65),   # gate/up, 15 groups of K: one row past the first 64-row block
    (1920, 15, 12160, 1024, 127),  # partial last row, 1520 weight tiles in blocks of 12
    (8192, 64, 1024, 256, 250),    # qkv (192-column blocks) and wo (128-column blocks)
    (640, 5, 1280, 29568, 80),     # BF16 head, five of a block's eight row chunks
    (640, 5, 1280, 29568, 128),
])
def test_wide_gemm_matches_oracle(hidden, heads, ffn, vocab, rows):
    kw = dict(vocab_size=vocab, hidden_dim=hidden, ffn_dim=ffn, n_layers=1, n_heads=heads, n_kv_heads=1,
              max_seq_len=rows + 8, weight_format=A.W_INT4_G128, kv_format=A.KV_F16, lm_head_format=1)
    ref, hip = make_pair(seed=41, max_batch=1, max_rows=rows, **kw)
    ids = R.synth_tokens(41, rows, rows, vocab)
    gl, gh = hip.forward_with_cache_output(ids[None], [0])
    wl, wh = ref.kv(rows + 8).forward(ids, 0, nthreads=16)
    assert np.isfinite(gl).all()
    assert rel_rows(gl[0], wl).max() < TOL, rel_rows(gl[0], wl).max()
    assert rel_rows(gh[0], wh).max() < TOL, rel_rows(gh[0], wh).max()
    hip.close()
