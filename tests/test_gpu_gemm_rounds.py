"""Projections whose blocks take more than one dispatch round run the GEMM's wide tiles without
k-splits: parity of the whole forward with the oracle (QatLinear::forward,
quant/src/qat.rs:315-348) with a partial last row chunk.
Bar: logits and hidden states within 2e-3 relative per row, as for every quantised forward."""
import numpy as np
import pytest

import aarambh_hip as A
import refcpu as R
from gpu_util import make_pair, rel_rows

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.mark.parametrize("wf,hidden,heads,ffn,vocab,rows", [
    (A.W_INT8_ROW, 640, 5, 12160, 50304, 201),  # gate/up and head
    (A.W_BF16, 640, 5, 12288, 1024, 135),       # gate/up
    (A.W_INT4_G128, 640, 5, 1280, 50304, 33),   # BF16 head, one row past two chunks
    (A.W_INT4_G128, 384, 3, 24576, 256, 139),   # INT4 gate/up, short K
])
def test_many_round_gemm_matches_oracle(wf, hidden, heads, ffn, vocab, rows):
    kw = dict(vocab_size=vocab, hidden_dim=hidden, ffn_dim=ffn, n_layers=1, n_heads=heads, n_kv_heads=1,
              max_seq_len=rows + 8, weight_format=wf, kv_format=A.KV_F16, lm_head_format=1)
    ref, hip = make_pair(seed=43, max_batch=1, max_rows=rows, **kw)
    ids = R.synth_tokens(43, rows, rows, vocab)
    gl, gh = hip.forward_with_cache_output(ids[None], [0])
    wl, wh = ref.kv(rows + 8).forward(ids, 0, nthreads=16)
    assert np.isfinite(gl).all()
    assert rel_rows(gl[0], wl).max() < TOL, rel_rows(gl[0], wl).max()
    assert rel_rows(gh[0], wh).max() < TOL, rel_rows(gh[0], wh).max()
    hip.close()
