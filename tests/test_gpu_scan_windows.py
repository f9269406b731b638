"""The exact sequential sums of the acceptance kernel take whole 512-value windows of a row at
once where the running sum stays in one binade: parity with the oracle's left-to-right sums
(sampler.rs:280-347, speculative.rs:770-793) at the edges of windows and of the 8192-value
chunks, for rows of equal terms (every add a rounding tie or exact), terms over the whole
range of exp, excluded (-inf) logits and one dominating term.
Bar: accepted lengths, tokens and draws identical unless either side flags a near-tie."""
import numpy as np
import pytest
import torch

import aarambh_hip as A
import refcpu as R

pytestmark = pytest.mark.gpu


def rows(kind, rng, shape):
    if kind == "equal":
        return np.full(shape, -1.25, np.float32)
    if kind == "wide":
        return -rng.uniform(0, 120, shape).astype(np.float32)
    x = (rng.normal(0, 3, shape)).astype(np.float32)
    if kind == "masked":
        x[rng.random(shape) < 0.7] = -np.inf
        x[..., 0] = 0.5
    if kind == "peak":
        x[..., shape[-1] // 2] = 60.0
    return x


@pytest.mark.parametrize("V", [1, 9, 511, 512, 513, 8191, 8192, 8193, 17001])
def test_window_edges_match_sequential_sums(V):
    m = A.HipModel(A.ModelConfig(vocab_size=128, hidden_dim=128, ffn_dim=128, n_layers=1, n_heads=1, n_kv_heads=1,
                                 max_seq_len=16), max_batch=1, max_rows=16)
    dev = torch.device("cuda:0")
    K, T = 2, 0.9
    first = last = 0
    for i, kind in enumerate(["normal", "equal", "wide", "masked", "peak"]):
        rng = np.random.default_rng([V, i])
        B = 6
        tgt = rows(kind, rng, (B, K + 1, V))
        drf = (tgt[:, :K] + np.where(np.isfinite(tgt[:, :K]), rng.normal(0, 1, (B, K, V)), 0)).astype(np.float32)
        toks = np.where(np.isfinite(drf), drf, -1e9).argmax(-1).astype(np.uint32)
        # the resampled or bonus draw lies in the first window, in the last one and between (a draw
        # within 1e-6 of a partial sum is flagged and not compared, so none is smaller than 1e-3)
        u = np.array([[0.999, 0.5, 0.9999], [1e-7, 0.3, 0.9997], [0.7, 0.95, 1e-3], [0.9999, 2e-3, 0.5],
                      [0.02, 0.9998, 2e-3], [1e-7, 1e-7, 0.0015]], np.float32)
        for top_p in (0.0, 0.9):
            s = A.Sampler.top_k_top_p(T, top_p=top_p)
            t = lambda a: torch.from_numpy(a).to(dev)
            out = m.accept_sample(t(tgt), t(drf), t(toks.astype(np.int32)), s, True, uniforms=t(u))
            out = {k: v.cpu().numpy() for k, v in out.items()}
            try:
                ref = R.accept_batch(tgt, drf, toks, R.sampler(temperature=T, top_p=top_p), True, uniforms=u)
            except ValueError:  # a distribution the reference refuses (its f32 sum is not within 1e-4 of 1)
                assert out["status"].any(), (kind, top_p, out)
                continue
            assert not out["status"].any(), (kind, top_p, out)
            flagged = (ref["flags"] != 0) | (out["flags"] != 0)
            same = (out["accept_len"] == ref["accept_len"]) & (out["token"] == ref["token"]) & (out["draws"] == ref["draws"])
            assert (same | flagged).all(), (kind, top_p, out, ref)
            assert (~flagged).sum() >= 3, (kind, top_p, ref)
            first += int((~flagged & (out["token"] < 512)).sum())
            last += int((~flagged & (out["token"] >= V - 512)).sum())
    assert first >= 12 and last >= 6, (first, last)  # crossings in the first and the last window that were compared
    m.close()
