"""Prompt chunks of more than 32 rows append their keys and values with a launch of their
own before the attention (inference/src/engine.rs:300-307 prefills in such chunks): parity
with the oracle at the edges of its 32-token cache blocks and 16-row query tiles.
Bar: logits and hidden states within 2e-3 relative per row, as for every quantised forward."""
import numpy as np
import pytest

import aarambh_hip as A
import refcpu as R
from gpu_util import make_pair, rel_rows

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.mark.parametrize("kvfmt", [A.KV_INT8, A.KV_F16])
@pytest.mark.parametrize("S,lens", [(32, [0, 20]),        # largest forward that appends in the attention
                                    (33, [0, 31]),        # smallest chunk; two blocks, and three
                                    (65, [1, 255, 256]),  # one row past two blocks; ends in a new chunk of tokens
                                    (100, [700]),         # several token chunks per query tile
                                    (128, [32, 0])])
def test_prompt_chunk_matches_oracle(kvfmt, S, lens):
    kw = dict(vocab_size=1024, hidden_dim=512, ffn_dim=512, n_layers=2, n_heads=4, n_kv_heads=2, max_seq_len=840,
              weight_format=A.W_INT8_ROW, kv_format=kvfmt, lm_head_format=1)
    n = len(lens)
    ref, hip = make_pair(seed=31, max_batch=n, max_rows=n * S, **kw)
    kvs = []
    for b, L in enumerate(lens):
        kv = ref.kv(840)
        if L:
            hip.kv_fill_synthetic(b, L, seed=60 + b)
            kv.fill_synthetic(60 + b, L)
        kvs.append(kv)
    # the chunk, then three rows that read it back from the cache
    for step, rows in enumerate((S, 3)):
        ids = R.synth_tokens(31, step, n * rows, 1024).reshape(n, rows)
        pos = [L + S * step for L in lens]
        gl, gh = hip.forward_with_cache_output(ids, pos)
        for b in range(n):
            wl, wh = kvs[b].forward(ids[b], pos[b], nthreads=16)
            assert np.isfinite(gl[b]).all()
            assert rel_rows(gl[b], wl).max() < TOL, (step, lens[b], rel_rows(gl[b], wl).max())
            assert rel_rows(gh[b], wh).max() < TOL, (step, lens[b], rel_rows(gh[b], wh).max())
    hip.close()
