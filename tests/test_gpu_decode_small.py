"""Decode steps of small models to the bit of the oracle at the edges of their own kernels: the attention in one launch
(contexts of up to 1024 positions, and of up to 64 Ki keys a head), and the FFN's activation quantized in w2's GEMV."""
import numpy as np
import pytest

import oracle_lib as ol
from paths import package

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def steps(cfg, prompt, count, seed):
    """`count` steps after a prompt of `prompt` tokens: every step's logits"""
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=seed), seed=seed + 1)
    cos, sin = package().rope_tables(cfg.seq_len, cfg.head_size, 10000.0, cfg.rotary)
    tokens = [int(t) for t in np.random.default_rng(seed).integers(0, cfg.vocab_size, size=prompt + count)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=1100)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=1100)
    if prompt:
        ref.run(tokens[:prompt], 0, False)
        eng.forwardMany(tokens[:prompt], 0)
    for pos in range(prompt, prompt + count):
        ref.run([tokens[pos]], pos, True)
        eng.forward(tokens[pos], pos, True)
        assert same_bits(eng.logits(), ref.logits()), pos
    eng.release()
    ref.close()


@pytest.mark.parametrize("half_kv", [0, 1])
@pytest.mark.parametrize("head_size,heads,kv_heads,prompt,count", [
    (48, 4, 4, 0, 9),        # the first positions: no whole four, a tail of every length
    (16, 8, 2, 253, 8),      # across a wave's positions and a four's thread
    (64, 4, 1, 1020, 8),     # the last positions of the one launch and the first past it
    (96, 2, 2, 680, 6),      # the keys' bound: 682 positions of 96 in float16
    (96, 2, 2, 509, 6),      # and 512 in float32
    (128, 4, 2, 509, 6),     # 512 of 128
    (256, 1, 1, 253, 6),     # 256 of 256
])
def test_attention_steps(head_size, heads, kv_heads, prompt, count, half_kv):
    cfg = ol.config(dim=heads * head_size, hidden_dim=96, n_layers=2, n_heads=heads, n_kv_heads=kv_heads,
                    head_size=head_size, vocab_size=96, seq_len=1056, shared_classifier=1, half_kv=half_kv)
    steps(cfg, prompt, count, seed=head_size)


@pytest.mark.parametrize("six", [0, 1])
@pytest.mark.parametrize("arch", ["llama", "gpt2"])
@pytest.mark.parametrize("hidden", [64, 1056, 4096, 4160])
def test_activation_in_the_down_projection(hidden, arch, six):
    """4096 is the widest row a one-token GEMV takes float32 values for; 1056 (int6: not an even number of groups)"""
    cfg = ol.config(dim=128, hidden_dim=hidden, n_layers=2, n_heads=4, n_kv_heads=4, head_size=32, vocab_size=96,
                    seq_len=32, shared_classifier=1, six=six, arch=arch)
    steps(cfg, 3, 4, seed=hidden)
