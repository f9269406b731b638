"""Prompt chunks over an fp16 cache: short ones append their keys and values inside the attention
kernel, each query tile up to its own last row, longer ones and batches of them with a launch of
their own (inference/src/engine.rs:300-307 prefills in such chunks): parity with the oracle at the
lengths where the path changes, and no launch's time added at 33 rows.
Bar: logits and hidden states within 2e-3 relative per row, as for every quantised forward."""
import numpy as np
import pytest

import aarambh_hip as A
import refcpu as R
from gpu_util import make_pair, rel_rows

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.mark.parametrize("heads,kv,S,lens", [
    (4, 2, 96, [700]),                    # longest chunk that appends in the attention, three token chunks
    (4, 2, 97, [5]),
    (8, 8, 64, [0, 31, 257, 3, 64, 1]),   # 6 sequences x 8 kv heads x 4 tiles x 64 rows = 12 288
    (8, 8, 64, [0, 31, 257, 3, 64, 1, 90]),  # 14 336: with a launch
    (6, 2, 50, [250])])                   # query tiles of 16 rows that end inside a position
def test_f16_chunk_matches_oracle(heads, kv, S, lens):
    kw = dict(vocab_size=512, hidden_dim=heads * 128, ffn_dim=512, n_layers=2, n_heads=heads, n_kv_heads=kv, max_seq_len=840,
              weight_format=A.W_INT8_ROW, kv_format=A.KV_F16, lm_head_format=1)
    n = len(lens)
    ref, hip = make_pair(seed=37, max_batch=n, max_rows=n * S, **kw)
    kvs = []
    for b, L in enumerate(lens):
        c = ref.kv(840)
        if L:
            hip.kv_fill_synthetic(b, L, seed=70 + b)
            c.fill_synthetic(70 + b, L)
        kvs.append(c)
    # the chunk, then three rows that read it back from the cache
    for step, rows in enumerate((S, 3)):
        ids = R.synth_tokens(37, step, n * rows, 512).reshape(n, rows)
        pos = [L + S * step for L in lens]
        gl, gh = hip.forward_with_cache_output(ids, pos)
        for b in range(n):
            wl, wh = kvs[b].forward(ids[b], pos[b], nthreads=16)
            assert np.isfinite(gl[b]).all()
            assert rel_rows(gl[b], wl).max() < TOL, (step, lens[b], rel_rows(gl[b], wl).max())
            assert rel_rows(gh[b], wh).max() < TOL, (step, lens[b], rel_rows(gh[b], wh).max())
    hip.close()


def attention_us(m, rows, ctx):
    ids = R.synth_tokens(3, rows, rows, 512)[None]
    t = []
    for _ in range(12):
        m.prof_enable(True)
        m.forward_with_cache_output(ids, [ctx], want_logits=False, want_hidden=False)
        prof = m.prof_get()["attention"]
        t.append(1e3 * prof["ms"] / prof["launches"])
    return sorted(t)[4]


def test_f16_short_chunk_time():
    """33 rows pay for one more query tile, not for an append launch (15 us against 24)."""
    m = A.HipModel(A.ModelConfig(vocab_size=512, hidden_dim=2048, ffn_dim=512, n_layers=4, n_heads=16, n_kv_heads=4,
                                 max_seq_len=1100, weight_format=A.W_INT8_ROW, kv_format=A.KV_F16, lm_head_format=1),
                   max_batch=1, max_rows=64)
    m.init_synthetic(seed=3, std=0.02)
    m.kv_fill_synthetic(0, 1000, seed=4)
    a, b = attention_us(m, 32, 1000), attention_us(m, 33, 1000)
    print(a, b)
    assert b < 1.25 * a, (a, b)
    m.close()
