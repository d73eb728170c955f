"""Prompt attention to the bit of the oracle where its weighted values leave the four-waves-a-tile kernel of small grids
for the one-wave-a-tile kernel: every head size with heads enough for the larger grid, both cache types, and the same
shapes just below it. A second layer's keys and values follow from every token's attention in the first."""
import numpy as np
import pytest

import oracle_lib as ol
from paths import package

pytestmark = pytest.mark.gpu

# head size: kv heads (each its own query head) whose 512 tokens are over 384 blocks of the larger grid
HEADS = {16: 50, 32: 26, 48: 18, 64: 14, 96: 10, 128: 8, 256: 4}


@pytest.mark.parametrize("half_kv", [0, 1])
@pytest.mark.parametrize("head_size", sorted(HEADS))
@pytest.mark.parametrize("m", [512, 67])
def test_prompt_attention_bits(head_size, m, half_kv):
    heads = HEADS[head_size]
    cfg = ol.config(dim=heads * head_size, hidden_dim=64, n_layers=2, n_heads=heads, n_kv_heads=heads,
                    head_size=head_size, vocab_size=64, seq_len=544, shared_classifier=1, half_kv=half_kv)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=6), seed=7)
    cos, sin = ol.rope_tables(cfg.seq_len, cfg.head_size, 10000.0)
    tokens = [int(t) for t in np.random.default_rng(head_size).integers(0, cfg.vocab_size, size=m + 9)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=544)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=544)
    for at, n in ((0, 9), (9, m)):
        ref.run(tokens[at:at + n], at, False)
        eng.forwardMany(tokens[at:at + n], at)
    k, v = ref.kv(0, m + 9)
    kv = eng.keysAndValues(0, m + 9)
    assert np.array_equal(kv["keys"].view(np.uint32), k.reshape(-1).view(np.uint32))
    assert np.array_equal(kv["values"].view(np.uint32), v.reshape(-1).view(np.uint32))
    eng.release()
    ref.close()
