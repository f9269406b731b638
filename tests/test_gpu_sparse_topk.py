"""Sampled acceptance with a top-k beyond the compact path that keeps few values of a row: parity
with the oracle (sampler.rs:226-347, speculative.rs:770-793) on both sides of the line (one value
in 75) where the scans' producers change.
Bar: accepted lengths, tokens and draws identical unless either side flags a near-tie."""
import numpy as np
import pytest
import torch

import aarambh_hip as A
import refcpu as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [82500, 82501, 76800])  # 82501 // 75 = 1100
@pytest.mark.parametrize("top_k,top_p", [(1099, 0.0), (1100, 0.9), (1025, 0.0)])
def test_sparse_topk_matches_oracle(V, top_k, top_p):
    m = A.HipModel(A.ModelConfig(vocab_size=128, hidden_dim=128, ffn_dim=128, n_layers=1, n_heads=1, n_kv_heads=1,
                                 max_seq_len=16), max_batch=1, max_rows=16)
    dev = lambda a: torch.from_numpy(a).to("cuda:0")
    B, K, T = 6, 2, 0.8
    rng = np.random.default_rng([V, top_k])
    tgt = rng.normal(0, 3, (B, K + 1, V)).astype(np.float32)
    drf = (tgt[:, :K] + rng.normal(0, 1, (B, K, V))).astype(np.float32)
    toks = drf.argmax(-1).astype(np.uint32)
    u = rng.uniform(0.05, 0.95, (B, K + 1)).astype(np.float32)
    s = A.Sampler.top_k_top_p(T, top_k=top_k, top_p=top_p)
    out = m.accept_sample(dev(tgt), dev(drf), dev(toks.astype(np.int32)), s, True, uniforms=dev(u))
    out = {k: v.cpu().numpy() for k, v in out.items()}
    ref = R.accept_batch(tgt, drf, toks, R.sampler(temperature=T, top_k=top_k, top_p=top_p), True, uniforms=u)
    assert not out["status"].any(), out
    flagged = (ref["flags"] != 0) | (out["flags"] != 0)
    same = (out["accept_len"] == ref["accept_len"]) & (out["token"] == ref["token"]) & (out["draws"] == ref["draws"])
    assert (same | flagged).all() and (~flagged).sum() >= 4, (out, ref)
    m.close()
