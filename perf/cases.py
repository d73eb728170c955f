"""The work a program gives the engine: quantized matmuls through hk_quantize_x / hk_matmul, prompts and conversation
turns through forwardMany and forward, answers through generateMany. A case is a dict of plain values; `listed` names
the fixed ones, `draw` makes more of the same ranges, `prepare` is what a program holds before the call, `run` is the
call, `work` its unavoidable bytes and operations, `tolerance` how far another correct implementation may lie from it,
`exact` the same result in 64 bits by plain torch.

Weights are synthetic in quantize.py's layout (N(0, 0.02), groups of 32), activations N(0, 1), prompts random ids.
"""
import ctypes
import importlib
import math

import numpy as np
import torch

GROUP = 32

# The shapes of the repository's benchmark and tests. `layers` is the depth of the whole model; a case may take fewer
# (a block of layers that is still larger than the 256 MB last-level cache) where the whole model adds only repetition.
MODELS = {
    "llama3-8b": dict(dim=4096, hidden_dim=14336, n_layers=32, n_heads=32, n_kv_heads=8, head_size=128,
                      vocab_size=128256, seq_len=4096, shared_classifier=0, half_kv=0, theta=500000.0),
    "qwen25-7b-int6": dict(dim=3584, hidden_dim=18944, n_layers=28, n_heads=28, n_kv_heads=4, head_size=128,
                           vocab_size=152064, seq_len=32768, shared_classifier=0, six=1, qkv_bias=1, half_kv=0,
                           rms_norm_eps=1e-6, theta=1000000.0),
    "llm150m": dict(dim=512, hidden_dim=2048, n_layers=12, n_heads=8, n_kv_heads=8, head_size=64, vocab_size=99487,
                    seq_len=1024, shared_classifier=1, half_kv=1, theta=10000.0),
    "stories15m": dict(dim=288, hidden_dim=768, n_layers=6, n_heads=6, n_kv_heads=6, head_size=48, vocab_size=32000,
                       seq_len=256, shared_classifier=1, half_kv=1, theta=10000.0),
    "gpt2-small": dict(dim=768, hidden_dim=3072, n_layers=12, n_heads=12, n_kv_heads=12, head_size=64,
                       vocab_size=50257, seq_len=1024, shared_classifier=1, half_kv=1, arch=1, theta=10000.0),
}
# the largest piece of a prompt a program hands over at once, and the steps of an answer it asks for at once
PROMPT_BLOCK, TOKEN_BLOCK, WINDOW, STOPS = 2048, 16, 64, [1]


def listed():
    return [
        # the standalone matmul: one layer's projections of one token (a decode step's matmul), of a short prompt and
        # of a prompt pass; a call a layer, each with its own weights, as a model makes them
        dict(name="matmul-token", kind="matmul", tokens=1, rows=4096, k=4096, bias=64, six=0, layers=16),
        dict(name="matmul-16", kind="matmul", tokens=16, rows=14336, k=4096, bias=64, six=0, layers=4),
        dict(name="matmul-512", kind="matmul", tokens=512, rows=14336, k=4096, bias=64, six=0, layers=1),
        # a greedy answer of the whole 8B model after a 2048-token prompt, sixteen tokens a call
        dict(name="answer-8b", kind="answer", model="llama3-8b", layers=32, start=2048, steps=16, temperature=0.0,
             topp=1.0, penalty=1.0),
        # reading a 2048-token prompt up to the first token's logits
        dict(name="prompt-8b", kind="prompt", model="llama3-8b", layers=4, start=0, tokens=2048, relaxed=1),
        # the next message of a conversation: a few dozen tokens after a context that is already cached
        dict(name="turn-8b", kind="prompt", model="llama3-8b", layers=4, start=1500, tokens=37, relaxed=1),
        # 6-bit weights, q/k/v biases, seven query heads a key head: a prompt of no round length
        dict(name="prompt-qwen", kind="prompt", model="qwen25-7b-int6", layers=4, start=0, tokens=1001, relaxed=1),
        # a sampled answer deep in a long context
        dict(name="answer-qwen-long", kind="answer", model="qwen25-7b-int6", layers=4, start=20003, steps=16,
             temperature=0.8, topp=1.0, penalty=1.1),
        # a small model whose weights stay in the caches: its prompt, with a float16 cache
        dict(name="prompt-150m", kind="prompt", model="llm150m", layers=12, start=0, tokens=512, relaxed=1),
        # the same in the plain order (bias 0), which a host without relaxed SIMD asks for
        dict(name="prompt-150m-plain", kind="prompt", model="llm150m", layers=12, start=0, tokens=301, relaxed=0),
        # the smallest model: a sampled answer with a nucleus and the repetition penalty, launches and latency
        dict(name="answer-15m", kind="answer", model="stories15m", layers=6, start=32, steps=48, temperature=0.8,
             topp=0.9, penalty=1.1),
        # the GPT-2 form (LayerNorm, learned positions, GELU, a bias after every matrix)
        dict(name="prompt-gpt2", kind="prompt", model="gpt2-small", layers=12, start=0, tokens=200, relaxed=1),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["matmul", "prompt", "prompt", "answer"])
    if kind == "matmul":
        return dict(kind=kind, tokens=_log_int(rng, 1, 512), rows=_log_int(rng, 96, 14336),
                    k=GROUP * _log_int(rng, 3, 448), bias=rng.choice([64, 64, 64, 0]), six=rng.choice([0, 0, 1]),
                    layers=1)
    model = rng.choice(sorted(MODELS))
    shape = MODELS[model]
    wide = shape["dim"] > 1024
    layers = 4 if wide else shape["n_layers"]
    if kind == "prompt":
        relaxed = 1 if wide or rng.random() < 0.7 else 0
        most = min(PROMPT_BLOCK, shape["seq_len"] // 2) if relaxed else min(400, shape["seq_len"] // 2)
        start = rng.choice([0, _log_int(rng, 1, min(4000, shape["seq_len"] // 2 - 1))])
        return dict(kind=kind, model=model, layers=layers, start=start, tokens=_log_int(rng, 2, most),
                    relaxed=relaxed)
    steps = rng.randint(5, 48)
    temperature = rng.choice([0.0, 0.8, 1.0])
    # (flat logits, as random weights of the wide models give, hold no nucleus that a device sorts)
    topp = rng.choice([0.9, 0.95, 1.0]) if temperature > 0 and not wide else 1.0
    return dict(kind=kind, model=model, layers=layers, start=_log_int(rng, 8, min(24000, shape["seq_len"] - 64)),
                steps=steps, temperature=temperature, topp=topp, penalty=rng.choice([1.0, 1.1]))


# ---- what a program holds before the call


def _package():
    return importlib.import_module("pyodide-llm_amd")


def _generator(seed, stream):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + stream) % (1 << 62))


def _quantized(x, six):
    """quantize.py's int8 (or int6 in int8) values of [rows, k] float32 and their group scales"""
    rows, k = x.shape
    g = x.reshape(rows, k // GROUP, GROUP)
    scale = g.abs().amax(-1) / (31.0 if six else 127.0)
    inverse = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    q = torch.round(g * inverse[..., None])
    if six:
        q = q.clamp(-32.0, 31.0) * 4.0
        scale = scale / 4.0
    return q.reshape(rows, k).to(torch.int8), scale


def _packed6(q):
    """a group's 32 six-bit values in 24 bytes: low nibbles of j and j + 16 in byte j, the top two bits of k, k + 8,
    k + 16 and k + 24 in byte 16 + k"""
    rows, k = q.shape
    b = (q.to(torch.int32) >> 2 & 63).reshape(rows, k // GROUP, 4, 8)
    nibbles = (b & 15).reshape(rows, k // GROUP, 2, 16)
    low = nibbles[:, :, 0] | nibbles[:, :, 1] << 4
    tops = b >> 4
    top = tops[:, :, 0] | tops[:, :, 1] << 2 | tops[:, :, 2] << 4 | tops[:, :, 3] << 6
    return torch.cat([low, top], -1).to(torch.uint8).reshape(rows, k // GROUP * 24)


def _matmul_inputs(case, seed, layer):
    """(quantized weights, their scales, the float32 activations) of one layer's call"""
    w = torch.randn(case["rows"], case["k"], device="cuda", generator=_generator(seed, 2 * layer)) * 0.02
    x = torch.randn(case["tokens"], case["k"], device="cuda", generator=_generator(seed, 2 * layer + 1))
    return (*_quantized(w, case["six"]), x)


def _config(case):
    shape = {k: v for k, v in MODELS[case["model"]].items() if k != "theta"}
    # the context a program opens the model with: the positions it will use, rounded up
    if case["model"] == "qwen25-7b-int6" and case["start"] < 4096:
        shape["seq_len"] = 8192
    shape["n_layers"] = case["layers"]
    shape["relaxed"] = case.get("relaxed", 1)
    return _package().config(**shape)


def _tokens(case, seed, count):
    rng = np.random.default_rng([seed, 7])
    ids = [int(t) for t in rng.integers(3, MODELS[case["model"]]["vocab_size"], size=count)]
    return [1] + ids[1:]


class _Chat:
    """an open model with a cached context, and what the next call is given"""


def _open(case, seed):
    pk = _package()
    cfg = _config(case)
    tensors, size = pk.places(cfg)
    cos, sin = pk.rope_tables(cfg.seq_len, cfg.head_size, MODELS[case["model"]]["theta"])
    engine = pk.open_synthetic(cfg, tensors, size, seed, cos, sin, max_block=PROMPT_BLOCK)
    if 0.0 < case.get("topp", 1.0) < 1.0:
        # logits as peaked as a trained model's (a nucleus of few tokens): the final norm's weights at 12
        ck = np.zeros(size, dtype=np.uint8)
        pk.hip_engine.check(pk.library().he_checkpoint_read(engine._h, 0, size, ctypes.c_void_p(ck.ctypes.data)))
        engine.release()
        at = tensors[pk.T["rms_final_weight"]].offset
        ck[at:at + 4 * cfg.dim] = np.full(cfg.dim, 12.0, dtype=np.float32).view(np.uint8)
        engine = pk.open_config(cfg, tensors, ck, cos, sin, max_block=PROMPT_BLOCK)
    return engine


def prepare(case, seed):
    if case["kind"] == "matmul":
        layers = []
        for layer in range(case["layers"]):
            q, scales, x = _matmul_inputs(case, seed, layer)
            layers.append(dict(w=_packed6(q) if case["six"] else q, ws=scales.contiguous(), x=x,
                               xq=torch.empty(x.shape, dtype=torch.int8, device="cuda"),
                               xs=torch.empty(x.shape[0], x.shape[1] // GROUP, device="cuda"),
                               y=torch.empty(x.shape[0], case["rows"], device="cuda")))
        return dict(case=case, layers=layers, pk=_package())
    chat = _Chat()
    chat.case = case
    chat.engine = _open(case, seed)
    if case["kind"] == "prompt":
        ids = _tokens(case, seed, case["start"] + case["tokens"])
        chat.fed = ids[case["start"]:]
        cached = ids[:case["start"]]
    else:
        ids = _tokens(case, seed, case["start"] + 1)
        cached, chat.history = ids[:-1], ids
        chat.randoms = [float(r) for r in np.random.default_rng([seed, 9]).random(case["steps"])]
    if cached:
        chat.engine.forwardMany(cached, 0)
    return chat


# ---- the call


def run(state):
    if isinstance(state, dict):
        return _run_matmul(state)
    if state.case["kind"] == "prompt":
        return _run_prompt(state)
    return _run_answer(state)


def _run_matmul(state):
    case, lib, check = state["case"], state["pk"].library(), state["pk"].hip_engine.check
    stream = torch.cuda.current_stream().cuda_stream
    for l in state["layers"]:
        check(lib.hk_quantize_x(l["xq"].data_ptr(), l["xs"].data_ptr(), l["x"].data_ptr(), case["tokens"], case["k"],
                                case["bias"], stream))
        check(lib.hk_matmul(l["y"].data_ptr(), l["xq"].data_ptr(), l["xs"].data_ptr(), l["w"].data_ptr(),
                            l["ws"].data_ptr(), case["tokens"], case["rows"], case["k"], case["bias"], case["six"],
                            stream))
    return [l["y"] for l in state["layers"]]


def _run_prompt(chat):
    """every token but the last through forwardMany, the last with its logits, as generate() feeds a prompt"""
    start, fed = chat.case["start"], chat.fed
    if len(fed) > 1:
        chat.engine.forwardMany(fed[:-1], start)
    chat.engine.forward(fed[-1], start + len(fed) - 1, True)
    return np.array(chat.engine.logits())


def _run_answer(chat):
    case, history, ids = chat.case, list(chat.history), []
    while len(ids) < case["steps"]:
        n = min(TOKEN_BLOCK, case["steps"] - len(ids))
        randoms = chat.randoms[len(ids):len(ids) + n] if case["temperature"] > 0 else []
        got = chat.engine.generateMany(history[-1], case["start"] + len(ids), history[-WINDOW:], len(history), n,
                                       case["temperature"], case["topp"], case["penalty"], randoms, STOPS)
        if got is None:
            raise RuntimeError("the engine left a step to its caller")
        ids += got
        history += got
        if got[-1] in STOPS:
            break
    return {"ids": np.array(ids, dtype=np.int32), "logits": np.array(chat.engine.logits())}


# ---- what the call cannot do without


def _row_bytes(k, six):
    return k * (0.75 if six else 1.0) + 4 * (k // GROUP)


def _layer_matrices(c):
    """(rows, k) of a layer's matrices"""
    q, kv = c.n_heads * c.head_size, c.n_kv_heads * c.head_size
    ffn = [(c.hidden_dim, c.dim), (c.dim, c.hidden_dim)] + ([] if c.arch else [(c.hidden_dim, c.dim)])
    return [(q, c.dim), (kv, c.dim), (kv, c.dim), (c.dim, q)] + ffn


def _step_work(c, start, tokens, logits):
    """bytes and operations of `tokens` tokens from position `start`: the weights read once, the tokens' embedding
    rows, the cached rows read once and the new ones written, the logits of `logits` of them"""
    row = lambda rows, k: rows * _row_bytes(k, c.six)  # noqa: E731
    weights = c.n_layers * sum(row(rows, k) for rows, k in _layer_matrices(c))
    values = c.n_layers * sum(rows * k for rows, k in _layer_matrices(c))
    kv = 2 * c.n_layers * c.n_kv_heads * c.head_size * (2 if c.half_kv else 4)
    positions = sum(start + t + 1 for t in range(tokens))
    classifier = row(c.vocab_size, c.dim) if logits else 0
    return (weights + classifier + tokens * row(1, c.dim) + (start + tokens) * kv + 4 * logits * c.vocab_size,
            2 * tokens * values + 2 * logits * c.vocab_size * c.dim
            + 4 * c.n_layers * c.n_heads * c.head_size * positions)


def work(case):
    if case["kind"] == "matmul":
        m, rows, k = case["tokens"], case["rows"], case["k"]
        return {"bytes": case["layers"] * (rows * _row_bytes(k, case["six"]) + 4 * m * k + 4 * m * rows),
                "flops": case["layers"] * 2 * m * rows * k}
    c = _config(case)
    if case["kind"] == "prompt":
        nbytes, ops = _step_work(c, case["start"], case["tokens"], 1)
        return {"bytes": nbytes, "flops": ops}
    # an answer's steps follow one another: each reads the weights and the cache again
    steps = [_step_work(c, case["start"] + i, 1, 1) for i in range(case["steps"])]
    return {"bytes": sum(b for b, _ in steps), "flops": sum(f for _, f in steps)}


def tolerance(case):
    """the engine's results are the reference's float32 operations in the reference's order, to the bit"""
    return "exact"


# ---- the same in 64 bits, by plain torch


def _activations64(x, bias):
    """quantize_x in float64: the values a group of 32 stands for"""
    g = x.reshape(x.shape[0], -1, GROUP)
    scale = g.abs().amax(-1, keepdim=True) / (63.0 if bias else 127.0)
    q = torch.where(scale > 0, torch.round(g / torch.where(scale > 0, scale, torch.ones_like(scale))),
                    torch.zeros_like(g))
    return (q * scale).reshape(x.shape)


def _widened64(q, scales):
    rows, k = q.shape
    return (q.reshape(rows, k // GROUP, GROUP).double() * scales.double()[..., None]).reshape(rows, k)


_MASK = (1 << 64) - 1


def _mix(z):
    z ^= z >> 30
    z = z * 0xBF58476D1CE4E5B9 & _MASK
    z ^= z >> 27
    z = z * 0x94D049BB133111EB & _MASK
    return z ^ z >> 31


def _signed(v):
    return v - (1 << 64) if v >= 1 << 63 else v


class _Checkpoint64:
    """the synthetic checkpoint's tensors in float64: the stated generator (a splitmix64 hash of seed, tensor and
    index, its four 16-bit quarters summed), quantize.py's rules, widened"""

    STREAMS = dict(embedding=0, wq=2, wk=3, wv=4, wo=5, w1=7, w2=8, w3=9, wcls=11, bq=12, bk=13, bv=14, positions=17,
                   ln_att=18, ln_ffn=19, ln_final=20, bo=21, b1=22, b2=23)

    def __init__(self, c, seed):
        self.c, self.seed = c, seed
        self.factor = float(np.float32(0.02 / math.sqrt(4.0 * (65536.0 * 65536.0 - 1.0) / 12.0)))

    def raw(self, name, index):
        key = _mix(self.seed * 0x9E3779B97F4A7C15 & _MASK ^ (self.STREAMS[name] * 0xD1B54A32D192ED03 & _MASK))
        z = index * _signed(0x9E3779B97F4A7C15) + _signed(key)
        for shift, times in ((30, 0xBF58476D1CE4E5B9), (27, 0x94D049BB133111EB), (31, 1)):
            z = z ^ (z >> shift & (1 << 64 - shift) - 1)
            z = z * _signed(times)
        total = (z & 0xFFFF) + (z >> 16 & 0xFFFF) + (z >> 32 & 0xFFFF) + (z >> 48 & 0xFFFF)
        return (total - 131070).float() * self.factor

    def rows(self, name, first, k):
        """the rows whose indices are `first` (an int64 tensor) of a matrix of row length k"""
        out = torch.empty(first.numel(), k, dtype=torch.float64, device="cuda")
        step = max(1, (1 << 25) // k)
        for at in range(0, first.numel(), step):
            index = first[at:at + step, None] * k + torch.arange(k, device="cuda")
            out[at:at + step] = _widened64(*_quantized(self.raw(name, index), self.c.six))
        return out

    def matrix(self, name, layer, rows, k):
        return self.rows(name, layer * rows + torch.arange(rows, device="cuda"), k)

    def vector(self, name, layer, n):
        return self.raw(name, layer * n + torch.arange(n, device="cuda")).double()


def _norm64(x, bias, eps):
    if bias is None:
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) + bias


def _rope64(x, theta):
    """interleaved pairs of [tokens, heads, size] turned by their positions (tables in float32, as handed over)"""
    t, _, size = x.shape
    freq = 1.0 / theta ** (torch.arange(0, size, 2, dtype=torch.float64, device="cuda") / size)
    angles = torch.arange(t, dtype=torch.float64, device="cuda")[:, None] * freq
    cos, sin = torch.cos(angles).float().double()[:, None], torch.sin(angles).float().double()[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)


def _attention64(q, k, v, c):
    t = q.shape[0]
    out = torch.empty_like(q)
    past = torch.ones(t, t, dtype=torch.bool, device="cuda").tril()
    for h in range(c.n_heads):
        j = h // (c.n_heads // c.n_kv_heads)
        s = (q[:, h] @ k[:, j].t()) / math.sqrt(c.head_size)
        out[:, h] = torch.softmax(s.masked_fill(~past, float("-inf")), -1) @ v[:, j]
    return out.reshape(t, -1)


def exact(case, seed):
    if case["kind"] == "matmul":
        out = []
        for layer in range(case["layers"]):
            q, scales, x = _matmul_inputs(case, seed, layer)
            out.append(_activations64(x.double(), case["bias"]) @ _widened64(q, scales).t())
        return out
    if case["kind"] == "answer":
        return None  # each token follows from the one before it, down to its last bit
    c, ids = _config(case), _tokens(case, seed, case["start"] + case["tokens"])
    ck, t = _Checkpoint64(c, seed), len(ids)
    bias = 64 if c.relaxed else 0
    ln = c.arch == 1
    at = torch.tensor(ids, device="cuda")
    x = ck.rows("embedding", at, c.dim)
    if ln:
        x = x + ck.rows("positions", torch.arange(t, device="cuda"), c.dim)
    q_dim, kv_dim = c.n_heads * c.head_size, c.n_kv_heads * c.head_size
    for l in range(c.n_layers):
        mul = lambda a, name, rows: a @ ck.matrix(name, l, rows, a.shape[1]).t()  # noqa: E731
        a = _activations64(_norm64(x, ck.vector("ln_att", l, c.dim) if ln else None, c.rms_norm_eps), bias)
        q, k, v = mul(a, "wq", q_dim), mul(a, "wk", kv_dim), mul(a, "wv", kv_dim)
        if ln or c.qkv_bias:
            q, k, v = (y + ck.vector(name, l, y.shape[1]) for y, name in ((q, "bq"), (k, "bk"), (v, "bv")))
        q, k, v = (y.reshape(t, -1, c.head_size) for y in (q, k, v))
        if not ln:
            q, k = _rope64(q, MODELS[case["model"]]["theta"]), _rope64(k, MODELS[case["model"]]["theta"])
        if c.half_kv:
            k, v = k.float().half().double(), v.float().half().double()
        x = x + mul(_activations64(_attention64(q, k, v, c), bias), "wo", c.dim)
        if ln:
            x = x + ck.vector("bo", l, c.dim)
            a = _activations64(_norm64(x, ck.vector("ln_ffn", l, c.dim), 0.0), bias)
            h = mul(a, "w1", c.hidden_dim) + ck.vector("b1", l, c.hidden_dim)
            h = h / (1.0 + torch.exp(-2.0 * math.sqrt(2.0 / math.pi) * (h + 0.044715 * h ** 3)))
            x = x + mul(_activations64(h, bias), "w2", c.dim) + ck.vector("b2", l, c.dim)
        else:
            a = _activations64(_norm64(x, None, c.rms_norm_eps), bias)
            h = mul(a, "w1", c.hidden_dim)
            h = h / (1.0 + torch.exp(-h)) * mul(a, "w3", c.hidden_dim)
            x = x + mul(_activations64(h, bias), "w2", c.dim)
    last = _activations64(_norm64(x[-1:], ck.vector("ln_final", 0, c.dim) if ln else None, c.rms_norm_eps), bias)
    out = torch.empty(c.vocab_size, dtype=torch.float64, device="cuda")
    name, step = "embedding" if c.shared_classifier else "wcls", 16384
    for first in range(0, c.vocab_size, step):
        rows = torch.arange(first, min(first + step, c.vocab_size), device="cuda")
        out[rows] = (last @ ck.rows(name, rows, c.dim).t())[0]
    return out
