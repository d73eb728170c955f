"""Decode attention whose ordered sums run from registers (segments of 32 values, 16 a row of lanes), to the bit of the
oracle: counts whose sums end on, just before and just past a segment, a pass of 16 segments and a chunk of 192 blocks, up
to the long contexts that the chunked kernel takes, in float32 and float16, from the cache of one prompt; and the chunked
kernel as a replayed step launches it, sized for the model's longest context."""
import numpy as np
import pytest

import oracle_lib as ol
from paths import package

pytestmark = pytest.mark.gpu

# 4 * blocks + rest positions: blocks of four at the edges of a segment (32), a pass (512) and, past what the kernel that
# keeps every product in LDS takes (8192), of an odd and an even number of chunks (11 and 12 of 192 blocks), every rest
LONG = (8200, 8447, 8448, 8453, 9213, 9216, 9219, 9222, 10240)
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


# a context of 9216 positions: the chunked kernel's launch, whose blocks take the steps of the kernel that keeps every product
# in LDS up to 2816 positions (what its own LDS holds), then 4 and 5 chunks of 768 positions and a little more or less
REPLAYED = (3, 126, 2813, 2814, 2815, 2816, 2817, 2818, 3067, 3071, 3072, 3073, 3078, 3839, 3840, 3841, 3846)
# the longest context of whole chunks that the kernel's LDS holds: 7680 positions
LONGEST = (1, 7679, 7680, 7681, 8453)


@pytest.mark.parametrize("heads,kv_heads,head_size,half_kv", [(7, 1, 128, 0), (8, 1, 128, 1), (7, 1, 64, 1), (4, 4, 64, 0),
                                                              (2, 2, 96, 0), (3, 1, 96, 1), (4, 1, 256, 0), (2, 1, 256, 1),
                                                              (8, 2, 32, 0), (6, 2, 48, 1)])
def test_replayed_steps_of_a_long_context(heads, kv_heads, head_size, half_kv):
    replayed_steps(heads, kv_heads, head_size, half_kv, 9216, REPLAYED)


@pytest.mark.parametrize("half_kv", [0, 1])
def test_replayed_steps_of_the_longest_context(half_kv):
    replayed_steps(4, 2, 16, half_kv, 32768, LONGEST)


def replayed_steps(heads, kv_heads, head_size, half_kv, seq_len, counts):
    cfg = ol.config(dim=96, hidden_dim=64, n_layers=1, n_heads=heads, n_kv_heads=kv_heads, head_size=head_size, vocab_size=64,
                    seq_len=seq_len, shared_classifier=1, half_kv=half_kv)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=6), seed=7)
    cos, sin = ol.rope_tables(cfg.seq_len, cfg.head_size, 10000.0)
    tokens = [int(t) for t in np.random.default_rng(head_size).integers(0, cfg.vocab_size, size=max(counts))]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=512)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=512)
    eng.generateMany(tokens[0], 0, [], 0, 2, 0.0, 0.9, 1.0, [], [])  # the graph (its first step runs eagerly)
    at = 0
    for count in counts:
        for end in list(range(at + 512, count - 1, 512)) + [count - 1]:
            if end > at:
                ref.run(tokens[at:end], at, False)
                eng.forwardMany(tokens[at:end], at)
                at = end
        ref.run([tokens[at]], at, True)
        got = eng.generateMany(tokens[at], at, [], 0, 1, 0.0, 0.9, 1.0, [], [])
        at += 1
        assert np.array_equal(np.asarray(eng.logits()).view(np.uint32), ref.logits().view(np.uint32)), count
        assert got == [int(np.argmax(ref.logits()))], count
    eng.release()
    ref.close()
