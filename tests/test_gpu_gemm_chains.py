"""The matmuls of more tokens than the GEMV takes, to the bit of the oracle, at the edges of the GEMM's tiles and of the
rules that pick one: 16 x 16, 32 x 32 and 64 x 32 blocks with a lane chain a wave, the 64 x 128 blocks of full grids, and
the SwiGLU epilogue's 16, 32 and 48 tokens; both biases, int8 and int6, every number of groups past the fours."""
import ctypes

import numpy as np
import pytest

import gpu_lib as gl
import oracle_lib as ol
from paths import package
from test_gpu_kernels import activations, same_bits, weights

pytestmark = pytest.mark.gpu

# (rows, k, m): one row, one group; the last row and token of a tile and the first of the next; stages cut after each
# number of groups
SMALL = [(1, 32, 2), (16, 64, 15), (17, 288, 16), (33, 544, 17), (100, 480, 33)]
MIDDLE = [(544, 352, 250), (513, 512, 241)]       # over 512 blocks of 16 x 16, at most 256 of 32 x 32
LARGE = [(1090, 288, 260), (1100, 1120, 257)]     # over 256 blocks of 32 x 32
FULL = [(2590, 96, 1170), (2560, 288, 1169)]      # the 64 x 128 blocks (bias 64)


@pytest.mark.parametrize("bias", [64, 0])
@pytest.mark.parametrize("six", [0, 1])
@pytest.mark.parametrize("rows,k,m", SMALL + MIDDLE + LARGE + FULL)
def test_matmul_bits(rows, k, m, six, bias):
    w, ws = weights(rows, k, six)
    xq, xs = activations(m, k, bias)
    assert same_bits(gl.matmul(xq, xs, w, ws, rows, k, bias, six), ol.matmul(xq, xs, w, ws, rows, k, bias, six))


# the last grids (in blocks of 64 x 32) that stay, and the first that leave for the 64 x 128 ones: of 96 values 504 / 525, of 128
# 700 / 702, of 224 520 / 528, of 256 820 / 828, of 992 756 / 768; past one of those a CU of 96 none, of 128 1340 / 1344, of 160
# 1080 / 1088, of 640 1420 / 1424, of 1120 1268 / 1272
STAY = [(2688, 96, 384), (1600, 128, 896), (4160, 224, 256), (2624, 256, 640), (2304, 992, 672), (21440, 128, 100), (17280, 160, 100),
        (22720, 640, 128), (20288, 1120, 128)]
LEAVE = [(4800, 96, 224), (2496, 128, 576), (2112, 224, 512), (2944, 256, 576), (2048, 992, 768), (16448, 96, 65), (21504, 128, 128),
         (17408, 160, 128), (22784, 640, 128), (20352, 1120, 128)]


@pytest.mark.parametrize("six", [0, 1])
@pytest.mark.parametrize("rows,k,m", STAY + LEAVE)
def test_where_the_64_x_128_blocks_start(rows, k, m, six):
    w, ws = weights(rows, k, six)
    xq, xs = activations(m, k, 64)
    some = np.r_[0:rows - 64:7, rows - 64:rows]  # (the oracle's rows: every seventh, the last block's all)
    got = gl.matmul(xq, xs, w, ws, rows, k, 64, six)[:, some]
    assert same_bits(got, ol.matmul(xq, xs, w[some], ws[some], len(some), k, 64, six))


@pytest.mark.parametrize("m", [2, 6, 7, 8, 9])
def test_where_the_gemv_ends(m):
    """bias 0, 40 rows: the GEMV in one pass, and in passes of two where a row's products are long; 9 such tokens on the GEMM"""
    for k in (96, 14336):
        w, ws = weights(40, k, 0)
        xq, xs = activations(m, k, 0)
        assert same_bits(gl.matmul(xq, xs, w, ws, 40, k, 0, 0), ol.matmul(xq, xs, w, ws, 40, k, 0, 0)), k


@pytest.mark.parametrize("relaxed", [1, 0])
@pytest.mark.parametrize("six", [0, 1])
@pytest.mark.parametrize("hidden,m", [(96, 5), (2784, 16), (2784, 40), (4160, 40), (2784, 97)])
def test_swiglu_epilogue_bits(hidden, m, six, relaxed):
    """a prompt block whose w1 / w3 GEMM finishes the SwiGLU: the second layer's keys and values follow from every token's
    output of the first layer's"""
    cfg = ol.config(dim=288, hidden_dim=hidden, n_layers=2, n_heads=6, n_kv_heads=6, head_size=48, vocab_size=320,
                    seq_len=128, shared_classifier=0, six=six, relaxed=relaxed)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=4), seed=5)
    cos, sin = ol.rope_tables(cfg.seq_len, cfg.head_size, 10000.0)
    tokens = [int(t) for t in np.random.default_rng(m).integers(0, cfg.vocab_size, size=m)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=128)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=128)
    ref.run(tokens, 0, False)
    eng.forwardMany(tokens, 0)
    kv, (k, v) = eng.keysAndValues(0, m), ref.kv(0, m)
    assert same_bits(kv["keys"], k.reshape(-1)) and same_bits(kv["values"], v.reshape(-1))
    eng.release()
    ref.close()


@pytest.mark.parametrize("arch,m", [("gpt2", 17), ("neox", 100), ("gpt2", 1024)])
def test_layer_norm_forms_epilogues(arch, m):
    """GPT-2's and GPT-NeoX's prompt layer: q/k/v finished in the GEMM (no rotation; part of each head turned), the biases
    after wo and w2, the GELU in the GEMM and, in a grid that the 64 x 128 blocks take (1024 tokens), on its own"""
    extra = dict(rotary=16, parallel_residual=1) if arch == "neox" else {}
    cfg = ol.config(dim=768, hidden_dim=3072, n_layers=2, n_heads=12, n_kv_heads=12, head_size=64, vocab_size=64,
                    seq_len=1024, shared_classifier=1, half_kv=1, arch=arch, **extra)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=8), seed=9)
    cos, sin = package().rope_tables(cfg.seq_len, cfg.head_size, 10000.0, cfg.rotary)
    tokens = [int(t) for t in np.random.default_rng(m).integers(0, cfg.vocab_size, size=m)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=1024)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=1024)
    ref.run(tokens, 0, False)
    eng.forwardMany(tokens, 0)
    kv, (k, v) = eng.keysAndValues(0, m), ref.kv(0, m)
    assert same_bits(kv["keys"], k.reshape(-1)) and same_bits(kv["values"], v.reshape(-1))
    eng.release()
    ref.close()


@pytest.mark.parametrize("six", [0, 1])
def test_biases_of_full_grids(six):
    """GPT-2's wo and w2 with a residual add and a bias where the 64 x 128 blocks take them (4096 rows, 1024 tokens)"""
    cfg = ol.config(dim=4096, hidden_dim=256, n_layers=2, n_heads=16, n_kv_heads=16, head_size=256, vocab_size=64,
                    seq_len=1024, shared_classifier=1, half_kv=1, arch="gpt2", six=six)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=8), seed=9)
    cos, sin = package().rope_tables(cfg.seq_len, cfg.head_size, 10000.0, cfg.rotary)
    tokens = [int(t) for t in np.random.default_rng(six).integers(0, cfg.vocab_size, size=1024)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=1024)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=1024)
    ref.run(tokens, 0, False)
    eng.forwardMany(tokens, 0)
    kv, (k, v) = eng.keysAndValues(1020, 4), ref.kv(1020, 4)
    assert same_bits(kv["keys"], k.reshape(-1)) and same_bits(kv["values"], v.reshape(-1))
    kv, (k, v) = eng.keysAndValues(0, 600), ref.kv(0, 600)
    assert same_bits(kv["keys"], k.reshape(-1)) and same_bits(kv["values"], v.reshape(-1))
    eng.release()
    ref.close()


def test_short_rows_finish_qkv():
    """q/k/v of a pass whose rows are so short that a plain matmul would leave the chains' blocks: the epilogue keeps them"""
    cfg = ol.config(dim=96, hidden_dim=96, n_layers=2, n_heads=32, n_kv_heads=32, head_size=64, vocab_size=64, seq_len=256,
                    shared_classifier=1)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=8), seed=9)
    cos, sin = package().rope_tables(cfg.seq_len, cfg.head_size, 10000.0)
    tokens = [int(t) for t in np.random.default_rng(1).integers(0, cfg.vocab_size, size=256)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=256)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=256)
    ref.run(tokens, 0, False)
    eng.forwardMany(tokens, 0)
    kv, (k, v) = eng.keysAndValues(0, 256), ref.kv(0, 256)
    assert same_bits(kv["keys"], k.reshape(-1)) and same_bits(kv["values"], v.reshape(-1))
    eng.release()
    ref.close()


def test_more_outputs_than_a_launch_has_threads():
    """bias 0, 131,072 rows x 131,136 tokens (69 GB of results): four outputs a thread are more than 2^32 threads"""
    rows, m, k = 1 << 17, (1 << 17) + 64, 32
    w, ws = weights(rows, k, 0)
    xq, xs = activations(m, k, 0)
    y = ctypes.c_void_p()
    gl.hip_check(gl.hip().hipMalloc(ctypes.byref(y), 4 * rows * m))
    try:
        args = [gl.upload(a) for a in (xq, np.ascontiguousarray(xs, np.float32), w, np.ascontiguousarray(ws, np.float32))]
        gl.check(package().library().hk_matmul(y, *(a.ptr for a in args), m, rows, k, 0, 0, None))
        gl.hip_check(gl.hip().hipDeviceSynchronize())
        row = np.zeros(rows, np.float32)
        for t in (0, 63, 70000, (1 << 17) - 1, 1 << 17, m - 1):
            gl.hip_check(gl.hip().hipMemcpy(ctypes.c_void_p(row.ctypes.data), ctypes.c_void_p(y.value + 4 * rows * t), row.nbytes, 2))
            assert same_bits(row, ol.matmul(xq[t:t + 1], xs[t:t + 1], w, ws, rows, k, 0, 0)[0]), t
    finally:
        gl.hip().hipDeviceSynchronize()
        gl.hip().hipFree(y)
