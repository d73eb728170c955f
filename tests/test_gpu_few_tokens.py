"""The matmuls of a few tokens on both sides of the lines between the GEMV (in passes where a launch does not take them all)
and the GEMM, to the bit of the oracle; the output projections of a short pass, which take the same rule with a residual add
and a bias; and that a few tokens against few long rows cost about what one does."""
import time

import numpy as np
import pytest

import gpu_lib as gl
import oracle_lib as ol
from paths import package
from test_gpu_kernels import activations, same_bits, weights

pytestmark = pytest.mark.gpu

# (rows, k, tokens): the shortest rows, the most tokens and the rows of a line, and just past each
INT8 = [(33, 576, 8), (33, 608, 8), (33, 608, 9), (1024, 640, 3), (1025, 640, 3), (1025, 1792, 6), (1025, 1824, 6),
        (1025, 1824, 7), (2049, 3040, 3), (2049, 3072, 3), (2049, 6976, 2), (2049, 7008, 3), (3073, 1024, 5), (3073, 1056, 5),
        (33, 8224, 7), (33, 8224, 8), (1030, 8224, 5), (1030, 8224, 6), (4100, 4096, 3), (4100, 4128, 3), (33, 28672, 5),
        (33, 28672, 6), (33, 40960, 6), (513, 40960, 6)]
INT6 = [(33, 832, 8), (33, 864, 8), (1025, 2016, 8), (1025, 2048, 8), (1030, 16416, 6), (1030, 16416, 7), (2049, 7008, 5),
        (2049, 7008, 6), (2049, 4064, 3), (2049, 4096, 3), (2049, 4608, 6), (2049, 4640, 6), (3073, 12000, 2), (3073, 12000, 3),
        (4100, 12000, 2), (4100, 16416, 2), (33, 18944, 8), (513, 18944, 8), (513, 20480, 8), (1025, 20480, 8)]
# bias 0: one pass of 8, then of 7, 3, 2 and 1
PLAIN = [(33, 288, 7), (33, 320, 7), (33, 320, 9), (1025, 640, 8), (33, 2048, 12), (33, 2048, 16), (33, 2048, 17),
         (1025, 2048, 9), (33, 4096, 9), (1025, 4096, 10), (1025, 4096, 12), (2050, 4096, 8), (33, 8192, 9), (33, 8192, 12), (1025, 8192, 6),
         (33, 14336, 8), (33, 14336, 9), (1025, 14336, 6), (33, 18944, 5), (33, 18944, 6), (3073, 18944, 2),
         (1025, 8192, 7), (1025, 8192, 9), (1025, 15360, 8), (33, 24576, 6), (1025, 24576, 5)]
# and past 4096 rows: one pass of 7 and 8, two of 3, 2 and 1, three of 1
PLAIN += [(4100, 2048, 7), (4100, 3104, 7), (4100, 4032, 8), (5130, 4096, 7), (4100, 8192, 4), (4100, 8192, 5), (4100, 10240, 4),
          (5130, 12288, 3), (7170, 12288, 3), (4100, 12288, 4), (4100, 14336, 4), (4100, 16352, 3), (10250, 18432, 2),
          (10240, 18944, 2), (10250, 18944, 2), (6150, 26016, 2)]


def check_matmul(rows, k, m, six, bias):
    w, ws = weights(rows, k, six)
    xq, xs = activations(m, k, bias)
    assert same_bits(gl.matmul(xq, xs, w, ws, rows, k, bias, six), ol.matmul(xq, xs, w, ws, rows, k, bias, six))


@pytest.mark.parametrize("six,rows,k,m", [(0, *c) for c in INT8] + [(1, *c) for c in INT6])
def test_relaxed_bits(rows, k, m, six):
    check_matmul(rows, k, m, six, 64)


@pytest.mark.parametrize("six", [0, 1])
@pytest.mark.parametrize("rows,k,m", PLAIN)
def test_plain_bits(rows, k, m, six):
    check_matmul(rows, k, m, six, 0)


@pytest.mark.parametrize("relaxed,m", [(1, 2), (1, 5), (1, 8), (0, 3), (0, 8), (0, 11)])
@pytest.mark.parametrize("six", [0, 1])
@pytest.mark.parametrize("arch", ["llama", "gpt2"])
def test_short_passes(arch, six, relaxed, m):
    """wo and w2 (rows of 1024 and 2080: a residual add, for GPT-2 a bias): the second layer's keys and values follow"""
    cfg = ol.config(dim=1024, hidden_dim=2080, n_layers=2, n_heads=8, n_kv_heads=8, head_size=128, vocab_size=96, seq_len=32,
                    shared_classifier=1, six=six, arch=arch, relaxed=relaxed)
    tensors, size = ol.places(cfg)
    ck = ol.vary_vectors(cfg, tensors, ol.synth_checkpoint(cfg, tensors, size, seed=2), seed=3)
    cos, sin = package().rope_tables(cfg.seq_len, cfg.head_size, 10000.0, cfg.rotary)
    tokens = [int(t) for t in np.random.default_rng(m).integers(0, cfg.vocab_size, size=m + 1)]
    ref = ol.Model(cfg, tensors, ck, cos, sin, max_block=32)
    eng = package().open_config(cfg, tensors, ck, cos, sin, max_block=32)
    for at, n in ((0, 1), (1, m)):
        ref.run(tokens[at:at + n], at, False)
        eng.forwardMany(tokens[at:at + n], at)
    kv, (k, v) = eng.keysAndValues(0, m + 1), ref.kv(0, m + 1)
    assert same_bits(kv["keys"], k.reshape(-1)) and same_bits(kv["values"], v.reshape(-1))
    eng.release()
    ref.close()


@pytest.mark.parametrize("rows,k,six,bias,few,many,most", [(96, 14336, 1, 64, 1, 2, 2.4), (1024, 14336, 0, 64, 1, 2, 2.4),
                                                           (1024, 4096, 1, 0, 6, 7, 2.4), (96, 14336, 0, 0, 2, 3, 3.0),
                                                           (1024, 28672, 1, 64, 4, 5, 1.85), (5120, 24576, 1, 0, 1, 2, 2.7)])
def test_few_tokens_cost_about_one_more(rows, k, six, bias, few, many, most):
    """Measured: 6.0 / 7.0 us, 7.2 / 10.2, 6.1 / 6.0, 11 / 22 (two passes of 2), 16.4 / 25.0 (of 4) and 29 / 59 (of 1), where the
    GEMM's block takes 19, 18, 17, 48, 35 and 94: under `most` times the time of `few`"""
    lib, check = package().library(), gl.check
    w, ws = (gl.upload(a) for a in weights(rows, k, six))

    def best(m):
        xq, xs = (gl.upload(a) for a in activations(m, k, bias))
        y = gl.Dev((m, rows), np.float32)
        times = []
        for _ in range(8):
            gl.hip_check(gl.hip().hipDeviceSynchronize())
            t = time.perf_counter()
            for _ in range(200):
                check(lib.hk_matmul(y.ptr, xq.ptr, xs.ptr, w.ptr, ws.ptr, m, rows, k, bias, six, None))
            gl.hip_check(gl.hip().hipDeviceSynchronize())
            times.append(time.perf_counter() - t)
        del xq, xs
        return min(times)

    assert best(many) < most * best(few)
