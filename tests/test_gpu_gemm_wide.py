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


# hidden, heads, ffn, vocab, rows, the projections that run in wide tiles (test_gemm_wide_rule.py)
CASES = [
    (1920, 15, 12160, 1024, 65, ["gate_up"]),   # 15 groups of K: one row past the first 64-row block
    (1920, 15, 12160, 1024, 127, ["gate_up"]),  # partial last row, 1520 weight tiles in blocks of 12
    (8192, 64, 1024, 256, 250, ["qkv", "wo"]),  # 192-column and 128-column blocks
    (640, 5, 1280, 29568, 80, ["head"]),        # five of a block's eight row chunks
    (640, 5, 1280, 29568, 128, ["head"]),
    (640, 5, 1280, 29568, 250, ["head"]),       # two row blocks, 231 column blocks, a partial last chunk
    (384, 3, 768, 21760, 383, ["head"]),        # three row blocks of 170 column blocks, normed rows in slices
]
# latent decoder: the fused q / kv_a / k_rope projection is a plain store of 10912 columns
LATENT = dict(vocab_size=256, hidden_dim=1024, n_layers=1, n_heads=56, max_seq_len=160, latent_dim=128, rope_dim=32,
              nope_dim=160, v_dim=32, n_experts=4, top_k=2, expert_dim=128, n_shared=1, expert_format=A.W_INT4_G128,
              attn_format=A.W_INT4_G128, lm_head_format=1, kv_format=A.KV_F16)
LATENT_ROWS = 250


@pytest.mark.parametrize("hidden,heads,ffn,vocab,rows,wide", CASES)
def test_wide_gemm_matches_oracle(hidden, heads, ffn, vocab, rows, wide):
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


def test_wide_store_matches_oracle():
    ref = R.LatModel(R.make_lat_config(**LATENT))
    ref.init_synthetic(11, 0.05)
    B, S = 2, LATENT_ROWS // 2
    hip = A.HipLatModel(A.LatConfig(**LATENT), max_batch=B, max_rows=LATENT_ROWS)
    hip.init_synthetic(11, 0.05)
    ids = R.synth_tokens(11, 1, LATENT_ROWS, LATENT["vocab_size"]).reshape(B, S)
    gl, gh = hip.forward_with_cache_output(ids, [0] * B)
    gaps = np.asarray(hip.router_gaps()).reshape(B, S)
    checked = 0
    for b in range(B):
        wl, wh = ref.kv(160).forward(ids[b], 0, nthreads=16)
        ok = gaps[b] >= 1e-4  # other rows may pick another expert of a near-tie
        checked += int(ok.sum())
        assert rel_rows(gl[b], wl)[ok].max() < TOL, rel_rows(gl[b], wl)[ok].max()
        assert rel_rows(gh[b], wh)[ok].max() < TOL, rel_rows(gh[b], wh)[ok].max()
    assert checked > LATENT_ROWS * 0.9, checked
    hip.close()
