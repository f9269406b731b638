"""Sampled acceptance at low temperatures, where most probabilities of a row are subnormal, zero or
quotients below 1e-30: parity with the oracle (filtered_probs and sample_from_probs,
sampler.rs:226-347; the residual, speculative.rs:770-793).
Bar: accepted lengths, tokens and draws identical unless either side flags a near-tie."""
import numpy as np
import pytest
import torch

import aarambh_hip as A
import refcpu as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [0.02, 0.05, 0.1, 0.3])
@pytest.mark.parametrize("V", [1000, 8193, 20000])
def test_low_temperature_matches_oracle(V, T):
    m = A.HipModel(A.ModelConfig(vocab_size=128, hidden_dim=128, ffn_dim=128, n_layers=1, n_heads=1, n_kv_heads=1,
                                 max_seq_len=16), max_batch=1, max_rows=16)
    dev = torch.device("cuda:0")
    B, K = 8, 3
    rng = np.random.default_rng([V, int(T * 100)])
    tgt = rng.normal(0, 3, (B, K + 1, V)).astype(np.float32)
    drf = (tgt[:, :K] + rng.normal(0, 0.3, (B, K, V))).astype(np.float32)
    toks = drf.argmax(-1).astype(np.uint32)
    u = rng.uniform(0.05, 0.95, (B, K + 1)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    unflagged = 0
    for kw in ({}, {"top_p": 0.9}, {"top_k": 1500}):
        out = m.accept_sample(t(tgt), t(drf), t(toks.astype(np.int32)), A.Sampler.top_k_top_p(T, **kw), True, uniforms=t(u))
        out = {k: v.cpu().numpy() for k, v in out.items()}
        ref = R.accept_batch(tgt, drf, toks, R.sampler(temperature=T, **kw), True, uniforms=u)
        assert not out["status"].any(), (kw, out)
        flagged = (ref["flags"] != 0) | (out["flags"] != 0)
        same = (out["accept_len"] == ref["accept_len"]) & (out["token"] == ref["token"]) & (out["draws"] == ref["draws"])
        assert (same | flagged).all(), (kw, out, ref)
        unflagged += int((~flagged).sum())
    assert unflagged >= 12, unflagged  # of 24
    m.close()


@pytest.mark.parametrize("T", [0.1, 0.9])
def test_non_finite_logits_match_oracle(T):
    """Infinite and NaN logits have probability 0 (sampler.rs:280-299)."""
    V, B, K = 3000, 6, 2
    m = A.HipModel(A.ModelConfig(vocab_size=128, hidden_dim=128, ffn_dim=128, n_layers=1, n_heads=1, n_kv_heads=1,
                                 max_seq_len=16), max_batch=1, max_rows=16)
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(9)
    tgt = rng.normal(0, 2, (B, K + 1, V)).astype(np.float32)
    drf = (tgt[:, :K] + rng.normal(0, 0.3, (B, K, V))).astype(np.float32)
    toks = drf.argmax(-1).astype(np.uint32)
    for x in (tgt, drf):
        hit = rng.random(x.shape)
        x[hit < 0.02] = np.inf
        x[(hit >= 0.02) & (hit < 0.04)] = np.nan
        x[(hit >= 0.04) & (hit < 0.3)] = -np.inf
    u = rng.uniform(0.05, 0.95, (B, K + 1)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    out = m.accept_sample(t(tgt), t(drf), t(toks.astype(np.int32)), A.Sampler.top_k_top_p(T), True, uniforms=t(u))
    out = {k: v.cpu().numpy() for k, v in out.items()}
    ref = R.accept_batch(tgt, drf, toks, R.sampler(temperature=T), True, uniforms=u)
    assert not out["status"].any(), out
    flagged = (ref["flags"] != 0) | (out["flags"] != 0)
    same = (out["accept_len"] == ref["accept_len"]) & (out["token"] == ref["token"]) & (out["draws"] == ref["draws"])
    assert (same | flagged).all() and (~flagged).sum() >= 3, (out, ref)
    m.close()
