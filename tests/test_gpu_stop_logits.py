"""The logits of a call that ends on a stop token, to the bit of the oracle's step: at the round's last step, where no replay
overwrites them, and before it, where the block that chose the token keeps them apart, for vocabularies that are not a
multiple of four and that take the block one round of its copy and several."""
import numpy as np
import pytest

import oracle_lib as ol
from paths import package
from steps import oracle_steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [67, 4098, 16384, 70001])
@pytest.mark.parametrize("temperature,topp,penalty", [(0.0, 0.9, 1.0), (0.0, 0.9, 1.2), (1.0, 1.0, 1.0), (0.7, 0.9, 1.1)])
def test_stopped_calls(vocab, temperature, topp, penalty):
    cfg = ol.config(dim=64, hidden_dim=96, n_layers=1, n_heads=4, n_kv_heads=4, head_size=16, vocab_size=vocab, seq_len=64,
                    shared_classifier=0)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=vocab), seed=1)
    if topp < 1.0:  # logits that are peaked enough for a nucleus the device sorts
        at = tensors[package().T["rms_final_weight"]].offset
        ck[at:at + 4 * cfg.dim] = np.full(cfg.dim, 30.0, np.float32).view(np.uint8)
    cos, sin = ol.rope_tables(cfg.seq_len, cfg.head_size, 10000.0)
    total = 24
    randoms = list(np.random.default_rng(vocab).random(total)) if temperature > 0.0 else [0.0] * total
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=16)
    history = [1, 5, 9]
    ref.run(history[:-1], 0, False)
    want, logits = oracle_steps(ref, list(history), len(history) - 1, total, temperature, topp, penalty, randoms)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=16)
    eng.forwardMany(history[:-1], 0)
    ends = [want.index(t) for t in dict.fromkeys(want)]
    assert ends[0] == 0
    for end in ends[:4] + [e for e in ends if e >= 14][:4]:
        for count in (end + 1, min(total, end + 3)):
            r = randoms[:count] if temperature > 0.0 else []
            for again in (0, 1):  # (a kind's first call runs its first step eagerly)
                got = eng.generateMany(history[-1], len(history) - 1, history, len(history), count, temperature, topp, penalty,
                                       r, [want[end]])
                assert got == want[:end + 1], (end, count, again)
                assert np.array_equal(np.asarray(eng.logits()).view(np.uint32), logits[end].view(np.uint32)), (end, count)
    eng.release()
    ref.close()
