"""Decode attention whose ordered sums run from registers (segments of 32 values, 16 a row of lanes), to the bit of the
oracle: counts whose sums end on, just before and just past a segment, a pass of 16 segments and a chunk of 256 blocks, up
to the long contexts that the chunked kernel takes, in float32 and float16, from the cache of one prompt."""
import numpy as np
import pytest

import oracle_lib as ol
from paths import package

pytestmark = pytest.mark.gpu

# 4 * blocks + rest positions: blocks of four at the edges of a segment (32), a pass (512) and, past what the kernel that
# keeps every product in LDS takes, of a chunk (256) and of two
LONG = (8200, 9213, 9216, 9219, 10240)
SHORT = (124, 127, 128, 133, 2047, 2048, 2052, 2176)


@pytest.mark.parametrize("half_kv", [0, 1])
@pytest.mark.parametrize("heads,kv_heads,head_size,counts", [(4, 2, 16, LONG), (2, 2, 48, (8200, 9217)), (2, 1, 64, SHORT)])
def test_decode_sums(heads, kv_heads, head_size, counts, half_kv):
    cfg = ol.config(dim=heads * head_size, hidden_dim=64, n_layers=1,
                    n_heads=heads, n_kv_heads=kv_heads, head_size=head_size, vocab_size=64, seq_len=(max(counts) & ~3) + 8,
                    shared_classifier=1, half_kv=half_kv)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=6), seed=7)
    cos, sin = ol.rope_tables(cfg.seq_len, cfg.head_size, 10000.0)
    tokens = [int(t) for t in np.random.default_rng(head_size).integers(0, cfg.vocab_size, size=max(counts) + 2)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=512)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=512)
    at = 0
    for count in counts:
        for end in list(range(at + 512, count - 1, 512)) + [count - 1]:
            if end > at:
                ref.run(tokens[at:end], at, False)
                eng.forwardMany(tokens[at:end], at)
                at = end
        ref.run([tokens[at]], at, True)
        eng.forward(tokens[at], at, True)
        at += 1
        assert np.array_equal(np.asarray(eng.logits()).view(np.uint32), ref.logits().view(np.uint32)), count
    eng.release()
    ref.close()
