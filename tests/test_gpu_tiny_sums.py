"""Sampled acceptance where the running sums of the softmax and the residual stay below 2^-103 over
most of a row (low temperatures, and a row's largest logit near its end): parity with the oracle's
left-to-right sums (sampler.rs:280-347, speculative.rs:770-793), in about the time of rows whose
sums are of ordinary size from the start.
Bar: accepted lengths, tokens and draws identical unless either side flags a near-tie."""
import time

import numpy as np
import pytest
import torch

import aarambh_hip as A
import refcpu as R

pytestmark = pytest.mark.gpu


def accept(m, dev, tgt, drf, toks, T, u):
    return m.accept_sample(dev(tgt), dev(drf), dev(toks.astype(np.int32)), A.Sampler.top_k_top_p(T), True, uniforms=dev(u))


@pytest.mark.parametrize("low", [-140.0, -104.0, -84.0])  # zero, subnormal and small normal terms
def test_tiny_sums(low):
    m = A.HipModel(A.ModelConfig(vocab_size=128, hidden_dim=128, ffn_dim=128, n_layers=1, n_heads=1, n_kv_heads=1,
                                 max_seq_len=16), max_batch=1, max_rows=16)
    dev = lambda a: torch.from_numpy(a).to("cuda:0")
    B, K, V, T = 4, 2, 32000, 0.1
    rng = np.random.default_rng(int(-low))
    times = []
    for peak in (V - 200, 40):  # the sums are tiny until the peak
        tgt = (T * rng.uniform(low - 6, low, (B, K + 1, V))).astype(np.float32)
        drf = (tgt[:, :K] + T * rng.uniform(-0.5, 0.5, (B, K, V))).astype(np.float32)
        # eight tokens hold the mass; the proposal is likely under the draft and hardly under the target
        tgt[..., peak:peak + 8] = T * rng.uniform(-1, 0, (B, K + 1, 8))
        drf[..., peak:peak + 8] = T * rng.uniform(-1, 0, (B, K, 8))
        toks = np.full((B, K), peak + 8, np.uint32)
        drf[..., peak + 8] = 0.0
        u = rng.uniform(0.1, 0.9, (B, K + 1)).astype(np.float32)
        out = {k: v.cpu().numpy() for k, v in accept(m, dev, tgt, drf, toks, T, u).items()}
        ref = R.accept_batch(tgt, drf, toks, R.sampler(temperature=T), True, uniforms=u)
        assert not out["status"].any(), out
        flagged = (ref["flags"] != 0) | (out["flags"] != 0)
        same = (out["accept_len"] == ref["accept_len"]) & (out["token"] == ref["token"]) & (out["draws"] == ref["draws"])
        assert (same | flagged).all() and not flagged.all(), (out, ref)
        args = [dev(x) for x in (tgt, drf, toks.astype(np.int32), u)]
        s = A.Sampler.top_k_top_p(T)
        t = []
        for _ in range(20):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            m.accept_sample(args[0], args[1], args[2], s, True, uniforms=args[3])
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        times.append(sorted(t)[5])
    # with the lanes of tiny windows added one by one, a row takes over a millisecond instead of 0.15
    assert times[0] < 2.0 * times[1], times
    m.close()
