"""Performance cases: the work that a program built on this library has it do, through the public entry points.

A case is a dict of plain values.  `listed()` names the representative ones, `draw(rng)` gives another one of the same ranges,
`prepare(case, seed)` makes what a program holds before the call (a model with its weights on the GPU, prompts), `run(state)`
is one pass of the call itself, `work(case)` the bytes and operations it cannot do without, `tolerance(case)` how far another
correct implementation of the same precision may be off.

The models are the published shapes this library is built for.  Weights are drawn like trained ones: matrices of standard
deviation 0.02, norm weights around one, and a final norm that gives the logits the spread of a trained model's (standard
deviation about 5, so that temperature and top-p have a distribution with a head and a tail to work on).
"""
import numpy as np

from llama2j_amd import BUFFER, TENSOR, Config, Transformer

# (dim, hidden_dim, n_layers, n_heads, n_kv_heads, vocab_size, seq_len, shared classifier)
SHAPES = {
    "stories15m": (288, 768, 6, 6, 6, 32000, 256, 1),
    "stories110m": (768, 2048, 12, 12, 12, 32000, 1024, 1),
    "llama2-7b": (4096, 11008, 32, 32, 32, 32000, 4096, 0),
    "llama2-13b": (5120, 13824, 40, 40, 40, 32000, 4096, 0),
    # the width and the grouped-query attention of the 70B shape, four of its eighty layers
    "llama2-70b-width": (8192, 28672, 4, 64, 8, 32000, 4096, 0),
}
SIGMA = 0.02
LOGIT_STD = 5.0


def listed():
    return [
        # One position with its logits on the host: a program that samples for itself, or scores a text, calls this per token.
        dict(name="forward-15m", kind="forward", model="stories15m", pos=100),
        # A short story from the smallest model, greedy: where latency is everything.
        dict(name="decode-15m", kind="decode", model="stories15m", prompt=8, new=56),
        # The reference's default way of generating (temperature 0.9, top-p 0.9) with the middle model.
        dict(name="sample-110m", kind="sample", model="stories110m", prompt=16, new=48, topp=0.9, prefill=0),
        # The headline use: greedy decode of the 7B shape behind a short prompt.
        dict(name="decode-7b", kind="decode", model="llama2-7b", prompt=16, new=32),
        # A chat turn: a prompt taken 32 positions per step (option "prefill"), then a sampled answer.
        dict(name="chat-7b", kind="sample", model="llama2-7b", prompt=150, new=24, topp=0.9, prefill=1),
        # A conversation that goes on deep in the context: the cache holds 3584 positions.
        dict(name="context-7b", kind="continue", model="llama2-7b", pos=3584, new=12),
        # The largest shape of the reference's configurations, greedy.
        dict(name="decode-13b", kind="decode", model="llama2-13b", prompt=8, new=16),
        # A server's batch: 32 requests with prompts of their own, greedy, the logits of every step kept.
        dict(name="batch-7b", kind="batch", model="llama2-7b", rows=32, prompt=20, new=10, temperature=0.0, topp=0.0),
        # A batch that is not full, sampled with plain top-p.
        dict(name="batch-sample-110m", kind="batch", model="stories110m", rows=13, prompt=12, new=20, temperature=0.9, topp=0.9),
        # Time to the first tokens of a question (a ragged length).
        dict(name="prefill-7b-short", kind="prefill", model="llama2-7b", tokens=77),
        # ... and of a document.
        dict(name="prefill-7b", kind="prefill", model="llama2-7b", tokens=1024),
        # A model brought up from fp32 host tensors, quantized on the device, up to its first logits.
        dict(name="load-15m", kind="load", model="stories15m", layers=6),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


# the most positions a drawn case may take of a model, so that it costs no more than the largest listed one
_MOST_STEPS = {"stories15m": 240, "stories110m": 300, "llama2-7b": 64, "llama2-13b": 32, "llama2-70b-width": 64}
_MOST_PREFILL = {"stories110m": 1000, "llama2-7b": 1000, "llama2-13b": 500, "llama2-70b-width": 1000}


def draw(rng):
    kind = rng.choice(["forward", "decode", "sample", "continue", "batch", "prefill", "prefill", "batch", "load"])
    if kind == "forward":
        model = rng.choice(sorted(SHAPES))
        return dict(kind=kind, model=model, pos=_log_int(rng, 1, SHAPES[model][6]) - 1)
    if kind == "continue":
        return dict(kind=kind, model=rng.choice(["stories110m", "llama2-7b"]), pos=_log_int(rng, 40, 1000), new=rng.randint(2, 16))
    if kind == "load":
        return dict(kind=kind, model=rng.choice(["stories15m", "stories110m"]), layers=rng.randint(1, 6))
    if kind == "prefill":
        model = rng.choice(sorted(_MOST_PREFILL))
        return dict(kind=kind, model=model, tokens=_log_int(rng, 2, _MOST_PREFILL[model]))
    if kind == "batch":
        sampled = rng.random() < 0.4
        model = "stories110m" if sampled else rng.choice(["stories110m", "llama2-7b", "llama2-70b-width"])
        return dict(kind=kind, model=model, rows=rng.randint(2, 32), prompt=_log_int(rng, 4, 24), new=rng.randint(2, 8),
                    temperature=rng.choice([0.6, 0.9]) if sampled else 0.0, topp=rng.choice([0.9, 1.0]) if sampled else 0.0)
    model = rng.choice(["stories15m", "stories110m", "llama2-7b", "llama2-13b"])
    steps = _log_int(rng, 12, _MOST_STEPS[model])
    prompt = rng.randint(1, steps // 2)
    if kind == "decode":
        return dict(kind=kind, model=model, prompt=prompt, new=steps - prompt)
    return dict(kind=kind, model=model, prompt=prompt, new=steps - prompt, topp=rng.choice([0.9, 1.0]),
                prefill=int(model != "stories15m" and rng.random() < 0.5))


def _shape(case):
    s = list(SHAPES[case["model"]])
    s[2] = case.get("layers", s[2])
    return s


def _norm_weights(rng, dim, n_layers):
    """Norm weights around one; the final ones scaled so that the logits' standard deviation is LOGIT_STD."""
    att = (1.0 + 0.1 * rng.standard_normal((n_layers, dim))).astype(np.float32)
    ffn = (1.0 + 0.1 * rng.standard_normal((n_layers, dim))).astype(np.float32)
    final = ((1.0 + 0.1 * rng.standard_normal(dim)) * (LOGIT_STD / (SIGMA * dim ** 0.5))).astype(np.float32)
    return att, ffn, final


def _model(case, seed, rng, options=None):
    shape = _shape(case)
    t = Transformer(Config(*shape), options=options)
    t.fill_synthetic(seed, SIGMA)
    for tensor, w in zip((TENSOR.RMS_ATT, TENSOR.RMS_FFN, TENSOR.RMS_FINAL), _norm_weights(rng, shape[0], shape[2])):
        t.upload_f32_quantize(tensor, w)
    t.finalize()
    return t


def _ids(rng, n):
    """Token ids of a text: no BOS, EOS or unknown among them."""
    return rng.integers(3, 32000, n).astype(np.int32)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "load":
        # what the checkpoint's file reader hands over: fp32 tensors in host memory
        dim, hidden, layers, heads, kv_heads, vocab, _, _ = shape = _shape(case)
        kvd = dim // heads * kv_heads
        sizes = {TENSOR.WQ: dim * dim, TENSOR.WK: kvd * dim, TENSOR.WV: kvd * dim, TENSOR.WO: dim * dim, TENSOR.W1: hidden * dim,
                 TENSOR.W2: dim * hidden, TENSOR.W3: hidden * dim}
        tensors = {t: (SIGMA * rng.standard_normal(layers * n, dtype=np.float32)) for t, n in sizes.items()}
        tensors.update(zip((TENSOR.RMS_ATT, TENSOR.RMS_FFN, TENSOR.RMS_FINAL), _norm_weights(rng, dim, layers)))
        return dict(kind=kind, shape=shape, tensors=tensors, embedding=SIGMA * rng.standard_normal((vocab, dim), dtype=np.float32))
    state = dict(case)
    state["t"] = t = _model(case, seed, rng, {"prefill": 1} if case.get("prefill") else None)
    if kind == "forward":
        state["token"] = int(_ids(rng, 1)[0])
        shape = SHAPES[case["model"]]
        if case["pos"] > 0:   # the cache rows of the positions before
            kvd = shape[0] // shape[3] * shape[4]
            n = min(case["pos"], 512)
            for layer in range(shape[2]):
                t.write_kv(layer, case["pos"] - n, rng.standard_normal((n, kvd), dtype=np.float32), rng.standard_normal((n, kvd), dtype=np.float32))
    elif kind == "continue":
        t.prefill(_ids(rng, case["pos"]), want_logits=False)
        state["token"] = int(_ids(rng, 1)[0])
    elif kind == "prefill":
        state["ids"] = _ids(rng, case["tokens"])
    elif kind == "batch":
        lengths = rng.integers(max(1, case["prompt"] * 2 // 3), case["prompt"] + 1, case["rows"])
        lengths[0] = case["prompt"]
        state["prompts"] = [_ids(rng, n) for n in lengths]
        state["seeds"] = rng.integers(1, 1 << 40, case["rows"])
    else:
        state["ids"] = _ids(rng, case["prompt"])
        state["seed"] = int(seed) + 1
    return state


def run(s):
    kind = s["kind"]
    if kind == "load":
        with Transformer(Config(*s["shape"])) as t:
            t.upload_f32(TENSOR.TOK_EMB, s["embedding"])
            for tensor, values in s["tensors"].items():
                t.upload_f32_quantize(tensor, values)
            t.finalize()
            return t.forward(1, 0)
    t = s["t"]
    if kind == "forward":
        return t.forward(s["token"], s["pos"])
    if kind == "decode":
        tokens, _ = t.decode_greedy(s["ids"], s["prompt"] + s["new"])
        return tokens, t.read(BUFFER.LOGITS)
    if kind == "sample":
        tokens, _ = t.decode_sample(s["ids"], s["prompt"] + s["new"], 0.9, s["topp"], s["seed"])
        return tokens, t.read(BUFFER.LOGITS)   # (the probabilities the last token was sampled from)
    if kind == "continue":
        token, tokens = s["token"], []
        for i in range(s["new"] - 1):
            token = t.forward_argmax(token, s["pos"] + i)
            tokens.append(token)
        return np.array(tokens), t.forward(token, s["pos"] + s["new"] - 1)
    if kind == "prefill":
        # the prompt, and the first position behind it, which attends to every cache row the prompt left
        logits, _ = t.prefill(s["ids"])
        return logits, t.forward(int(np.argmax(logits)), s["tokens"])
    tokens, _, logits = t.decode_sample_batch(s["prompts"], s["prompt"] + s["new"], s["temperature"], s["topp"], s["seeds"], want_logits=True)
    return tokens, logits


def _matrix_weights(shape):
    dim, hidden, layers, heads, kv_heads = shape[:5]
    kvd = dim // heads * kv_heads
    return layers * (2 * dim * dim + 2 * kvd * dim + 3 * dim * hidden)


def work(case):
    """Weights and cache rows read once per dependent step (264 bytes per 256 quantized weights, fp32 classifier and cache), two
    operations per weight and position."""
    shape, kind = _shape(case), case["kind"]
    dim, layers, vocab = shape[0], shape[2], shape[5]
    kvd = dim // shape[3] * shape[4]
    w = _matrix_weights(shape)
    body, cls, row = w * 264 / 256, 4.0 * vocab * dim, 8.0 * layers * kvd   # row: k and v of one position, all layers

    def positions(first, n):   # operations of n positions without the classifier
        return n * (2.0 * w + 4.0 * layers * dim * (first + (n + 1) / 2.0))

    def steps(first, n):       # n positions one after the other: everything is read for each
        return dict(bytes=n * (body + cls + 4.0 * dim) + row * n * (first + (n + 1) / 2.0), flops=positions(first, n) + n * 2.0 * vocab * dim)

    if kind == "load":
        return dict(bytes=2 * 4.0 * (w + vocab * dim) + body, flops=2.0 * w + 2.0 * vocab * dim)
    if kind == "forward":
        return steps(case["pos"], 1)
    if kind == "continue":
        return steps(case["pos"], case["new"])
    if kind == "prefill":
        n, last = case["tokens"], steps(case["tokens"], 1)
        return dict(bytes=body + cls + n * (4.0 * dim + row) + last["bytes"], flops=positions(0, n) + 2.0 * vocab * dim + last["flops"])
    if kind == "batch":
        # the prompts' positions are known: they need the weights once; every later step needs them again
        n, rows = case["prompt"] + case["new"], 16 if case["rows"] <= 16 else 32
        return dict(bytes=(case["new"] + 1) * (body + cls) + rows * (row * n * (n + 1) / 2.0 + 2 * 4.0 * n * vocab),
                    flops=rows * (positions(0, n) + n * 2.0 * vocab * dim))
    n = case["prompt"] + case["new"]
    if case.get("prefill"):   # whole steps of 32 prompt positions at once, the rest one after the other
        at_once = case["prompt"] // 32 * 32
        rest = steps(at_once, n - at_once)
        if at_once:
            rest = dict(bytes=rest["bytes"] + body + at_once * row, flops=rest["flops"] + positions(0, at_once))
        return rest
    return steps(0, n)


# Measured between two orders of the same sums (a prompt taken 32 positions at a time on the matrix cores against position by
# position, 33 to 700 positions, 24 tokens behind): the logits' relative error, their largest difference over the root mean
# square, and both again for sampled probabilities.  The deeper and wider shapes amplify the same rounding more.
_SPREAD = {
    "stories15m": (1.6e-6, 7e-6, 7e-6, 2.1e-5),
    "stories110m": (1.6e-6, 7e-6, 7e-6, 2.1e-5),
    "llama2-7b": (1.1e-5, 5e-5, 4.5e-5, 1.2e-4),
    "llama2-13b": (1.6e-5, 7e-5, 7.5e-5, 2.1e-4),
    "llama2-70b-width": (6.8e-6, 2.6e-5, 1.8e-5, 8e-5),
}


def tolerance(case):
    """Four times the measured spread; a token in a hundred may differ, where two candidates lie within it of each other."""
    rel, most, p_rel, p_most = _SPREAD[case["model"]]
    if case["kind"] == "sample":
        rel, most = p_rel, p_most
    return {"rel": 4 * rel, "max": 4 * most, "differ": 0.01}
