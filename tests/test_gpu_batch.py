"""Sixteen or thirty-two sequences at once (l2j_decode_greedy_batch, l2j_batch_matmul): the matrix-core path must give
every sequence what it gets alone.  Checked through the C ABI against the single-sequence path (itself pinned against the CPU oracle
in test_gpu_parity.py), against the oracle directly, and against float64 products of the dequantized weights."""
import numpy as np
import pytest

import llama2j_amd as l2j
from llama2j_amd import TENSOR
from llama2j_amd.binding import L2JError

pytestmark = pytest.mark.gpu

LOGIT_TOL = 1e-3   # per step: max |logit - oracle's| / max |oracle's logit|, the bar of the single-sequence path


def rel_err(got, want):
    return float(np.abs(got.astype(np.float64) - want).max() / np.abs(want).max())


def oracle_of(orc, shape, seed):
    m = orc.Model(dim=shape[0], hidden_dim=shape[1], n_layers=shape[2], n_heads=shape[3], n_kv_heads=shape[4],
                  vocab_size=shape[5], seq_len=shape[6], shared_weights=shape[7])
    m.fill_synth(seed, 0.02)
    return m


def check_against_oracle(m, prompt, steps, tokens, logits, what):
    """The oracle's own greedy loop from the same prompt: the same tokens (until it stops at token 1; the batch runs on), and at
    every one of those steps the batched path's logits within the bar of the oracle's."""
    m.reset()
    want_tok, want_logits, _ = m.generate_greedy(prompt, steps, want_logits=True)
    np.testing.assert_array_equal(tokens[:len(want_tok)], want_tok, err_msg=what)
    worst = max(rel_err(logits[pos], want_logits[pos]) for pos in range(len(want_tok)))
    assert worst < LOGIT_TOL, (what, worst)
    return worst

def same_until_a_tie(got, want, logits, what):
    """The batched path and the single-sequence path add the same products in different orders (their logits agree to a
    few 1e-6 of the largest), so a sequence may part ways where its two best logits lie that close together, and only
    there: the same tokens up to the first difference, and at that step the two tokens' logits (the batched path's) within
    1e-5 of the largest."""
    diff = np.flatnonzero(got != want)
    if diff.size == 0:
        return
    pos = int(diff[0])
    lg = logits[pos]
    gap = abs(float(lg[got[pos]]) - float(lg[want[pos]]))
    assert gap <= 1e-5 * float(np.abs(lg).max()), (what, pos, int(got[pos]), int(want[pos]), gap)


SHAPES = [
    (512, 1024, 4, 8, 8, 1008, 64, 1),      # head 64, shared classifier
    (512, 1024, 2, 8, 2, 1008, 64, 0),      # grouped-query attention: 8 heads on 2 kv heads
    (1024, 2816, 2, 8, 4, 2000, 96, 0),     # head 128, rows of 4 and 11 groups (an odd number of groups: a last slice of one)
    (512, 768, 2, 2, 2, 512, 40, 1),        # head 256
    (512, 1024, 2, 8, 2, 1008, 640, 0),     # 640 positions: the row slots of the attention kernel go round forty times
]


def dequantized(g, tensor, layer, rows, K):
    """One layer's matrix as float64, from the .quant bytes the library serialises (min, max big-endian, 256 codes)."""
    per = rows * K // 256
    raw = g.read_quant(tensor, layer * per, per).reshape(per, 264)
    hdr = raw[:, :8].copy().view(">f4").astype(np.float32)
    mn, mx = hdr[:, 0], hdr[:, 1]
    rm = ((mx - mn) / np.float32(255.0)).astype(np.float32)          # K/MatMul.java:137
    w = raw[:, 8:].astype(np.float32) * rm[:, None] + mn[:, None]    # K/MatMul.java:141
    return w.reshape(rows, K).astype(np.float64)


def test_matrix_core_product_matches_float64():
    shape = (1024, 2816, 2, 8, 4, 2000, 96, 0)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(7, 0.02)
    g.finalize()
    rng = np.random.default_rng(0)
    kvd = 1024 * 4 // 8
    for tensor, rows, K in ((TENSOR.WQ, 1024, 1024), (TENSOR.WK, kvd, 1024), (TENSOR.W1, 2816, 1024), (TENSOR.W2, 1024, 2816)):
        x = (rng.standard_normal((16, K)) * np.exp(rng.uniform(-3, 3, (16, 1)))).astype(np.float32)
        want = x.astype(np.float64) @ dequantized(g, tensor, 1, rows, K).T
        got, _ = g.batch_matmul(tensor, 1, x, rows)
        err = np.abs(got - want).max(axis=1) / np.abs(want).max(axis=1)      # per sequence
        assert err.max() < 5e-6, (int(tensor), float(err.max()))
    g.close()


@pytest.mark.parametrize("n_seq", [16, 32])
@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[2], SHAPES[3]])
def test_the_layers_of_a_step_in_one_launch_give_the_same(orc, shape, n_seq):
    """Option batch_fuse = 1 runs all layers of a step in one resident kernel with grid barriers (deferred rmsnorm scalars,
    its own attention phase): the tokens of the launch-per-phase step, and the oracle's logits within the same bar."""
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(shape[1] + n_seq)
    steps = shape[6]
    prompts = [rng.integers(2, shape[5], size=int(rng.integers(0, 9))).astype(np.int32) for _ in range(n_seq - 2)]
    want, _ = g.decode_greedy_batch(prompts, steps, n_seq=n_seq)
    g.set_option("batch_fuse", 1)
    got, logits = g.decode_greedy_batch(prompts, steps, n_seq=n_seq, want_logits=True)
    again, _ = g.decode_greedy_batch(prompts, steps, n_seq=n_seq)
    g.close()
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(again, got)
    m = oracle_of(orc, shape, 9)
    for b in (0, n_seq // 2, n_seq - 1):
        p = prompts[b] if b < len(prompts) else np.zeros(0, dtype=np.int32)
        check_against_oracle(m, p, steps, got[b], logits[:, b], "sequence %d against the oracle" % b)
    m.close()


@pytest.mark.parametrize("n_seq", [16, 32])
@pytest.mark.parametrize("shape", SHAPES)
def test_every_sequence_gets_what_it_gets_alone(orc, shape, n_seq):
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(shape[0] + shape[4] + n_seq)
    steps = shape[6]
    prompts = [rng.integers(2, shape[5], size=int(rng.integers(0, 9))).astype(np.int32) for _ in range(n_seq - 3)]   # three without a prompt
    got, sec = g.decode_greedy_batch(prompts, steps, n_seq=n_seq)
    assert got.shape == (n_seq, steps) and sec > 0
    got2, logits = g.decode_greedy_batch(prompts, steps, n_seq=n_seq, want_logits=True)   # (the same buffers and graph again)
    np.testing.assert_array_equal(got2, got)
    for b in range(n_seq):
        p = prompts[b] if b < len(prompts) else np.zeros(0, dtype=np.int32)
        g.reset()
        want, _ = g.decode_greedy(p, steps)          # stops after token 1; the batch runs on
        same_until_a_tie(got[b, :len(want)], want, logits[:, b], "sequence %d" % b)
        np.testing.assert_array_equal(got[b, :len(p)], p)
    # every sequence against the oracle as well: its tokens, and the logits of every step
    m = oracle_of(orc, shape, 9)
    worst = 0.0
    for b in range(n_seq):
        p = prompts[b] if b < len(prompts) else np.zeros(0, dtype=np.int32)
        worst = max(worst, check_against_oracle(m, p, steps, got[b], logits[:, b], "sequence %d against the oracle" % b))
    print("batched logits vs oracle: worst max|d|/max|logit| = %.3g over %d sequences x %d steps" % (worst, n_seq, steps), flush=True)
    # the context's own cache and loop state are untouched: a single decode after the batch is what it was before
    g.reset()
    again, _ = g.decode_greedy(prompts[0], steps)
    np.testing.assert_array_equal(again, got[0, :len(again)])
    m.close(); g.close()


@pytest.mark.parametrize("n_seq", [16, 32])
@pytest.mark.parametrize("hidden", [4096, 4352, 8448, 12544])
def test_products_of_one_to_four_tiles_per_workgroup(orc, hidden, n_seq):
    # W1 and W3 over one slice of 256: hidden / 16 tiles of 32 rows on 256 workgroups, the last round full or not
    test_every_sequence_gets_what_it_gets_alone(orc, (256, hidden, 1, 4, 4, 512, 40, 1), n_seq)


@pytest.mark.parametrize("n_seq", [16, 32])
@pytest.mark.parametrize("dim,hidden", [(256, 256), (256, 2048), (768, 2048), (1024, 2048), (1024, 2304), (1280, 2048)])
def test_swiglu_within_the_products_up_to_its_last_shape(orc, dim, hidden, n_seq):
    # SwiGLU at the end of W1 and W3, its digits at the beginning of W2: up to 4 groups of dim, 8 of hidden, 256 workgroups for W2 (1024, 2048); past
    # that a launch of its own
    test_every_sequence_gets_what_it_gets_alone(orc, (dim, hidden, 2, dim // 64, dim // 64, 512, 24, 1), n_seq)


@pytest.mark.parametrize("shape", [(768, 2048, 2, 12, 12, 1008, 24, 1), (512, 1280, 2, 8, 2, 1008, 24, 0), (1024, 2816, 2, 8, 4, 2000, 24, 0)])
def test_a_sequence_has_the_same_bits_among_sixteen_and_among_32(shape):
    """The products of up to sixteen vectors and those of up to 32 add a row up in the same order, so a sequence's logits, and with them
    what is sampled from them, do not depend on how many others there are."""
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(shape[1])
    prompts = [rng.integers(2, shape[5], size=b % 7).astype(np.int32) for b in range(32)]   # (the first has none: no prompt positions in common)
    want_tokens, want = g.decode_greedy_batch(prompts, shape[6], want_logits=True)
    for first in (0, 14):
        tokens, logits = g.decode_greedy_batch(prompts[first:first + 16], shape[6], want_logits=True)
        np.testing.assert_array_equal(tokens, want_tokens[first:first + 16])
        np.testing.assert_array_equal(logits.view(np.uint32), want[:, first:first + 16].view(np.uint32))
    g.close()


@pytest.mark.parametrize("dim,groups,wider", [(256, 1, 9), (512, 3, 9), (768, 4, 10), (512, 5, 9), (768, 6, 9), (256, 7, 10), (768, 8, 16), (1024, 8, 12)])
def test_hidden_rows_of_zeros_change_no_bit(dim, groups, wider):
    """The same layers with further rows of zeros in W1 and W3 and zeros behind the rows of W2, so many that SwiGLU is a launch of its own:
    the logits of every step have the same bits.  (Both widths cut a row into slices of as many groups.)"""
    n_layers, vocab, seq_len = 2, 512, 16
    rng = np.random.default_rng(dim + groups)
    weights = {t: 0.02 * rng.standard_normal((n_layers, 256 * groups, dim)).astype(np.float32) for t in (TENSOR.W1, TENSOR.W3)}
    weights[TENSOR.W2] = 0.02 * rng.standard_normal((n_layers, dim, 256 * groups)).astype(np.float32)
    prompts = [rng.integers(2, vocab, size=b % 5).astype(np.int32) for b in range(32)]
    want = None
    for width in (groups, wider):
        g = l2j.Transformer(l2j.Config(dim, 256 * width, n_layers, dim // 64, dim // 64, vocab, seq_len, 1))
        g.fill_synthetic(9, 0.02)
        for t, w in weights.items():
            pad = [(0, 0)] * 3
            pad[2 if t == TENSOR.W2 else 1] = (0, 256 * (width - groups))
            g.upload_f32_quantize(t, np.pad(w, pad))
        for t in (TENSOR.RMS_ATT, TENSOR.RMS_FFN, TENSOR.RMS_FINAL):
            g.upload_f32_quantize(t, np.ones(dim * (1 if t == TENSOR.RMS_FINAL else n_layers), dtype=np.float32))
        for t, rows in ((TENSOR.WQ, dim), (TENSOR.WK, dim), (TENSOR.WV, dim), (TENSOR.WO, dim)):
            g.upload_f32_quantize(t, 0.02 * np.random.default_rng(int(t)).standard_normal((n_layers, rows, dim)).astype(np.float32))
        g.upload_f32(TENSOR.TOK_EMB, 0.02 * np.random.default_rng(1).standard_normal((vocab, dim)).astype(np.float32))
        g.finalize()
        got = [g.decode_greedy_batch(prompts[:n], seq_len, want_logits=True) for n in (16, 32)]
        got.append((np.int32(0), g.prefill(np.arange(2, 2 + 11, dtype=np.int32))[0]))
        g.close()
        if want is None:
            want = got
        for (tokens, logits), (tokens1, logits1) in zip(got, want):
            np.testing.assert_array_equal(tokens, tokens1)
            np.testing.assert_array_equal(logits.view(np.uint32), logits1.view(np.uint32))


@pytest.mark.parametrize("heads", [8, 4, 2])
def test_scores_of_minus_infinity_weigh_nothing(heads):
    """A token whose keys are huge in one element of head 0 and whose queries are negative there: it scores -inf against itself and its
    like, and what is left is the softmax over the other rows, also where the first rows that a wave takes are all of its kind."""
    shape, head, huge, other = (512, 1024, 1, heads, heads, 64, 80, 0), 512 // heads, 3, 4
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    emb = np.random.default_rng(heads).standard_normal((64, 512), dtype=np.float32)
    emb[:, 0] = 0
    emb[[1, huge], 0] = 10.0   # (token 1 comes first)
    g.upload_f32(TENSOR.TOK_EMB, emb)
    for t in (TENSOR.RMS_ATT, TENSOR.RMS_FFN, TENSOR.RMS_FINAL):
        g.upload_f32_quantize(t, np.linspace(0.9, 1.1, 512, dtype=np.float32))
    for t, w in ((TENSOR.WK, 1e28), (TENSOR.WQ, -1e12)):
        m = 0.02 * np.random.default_rng(int(t)).standard_normal((512, 512), dtype=np.float32)
        m[head - 2] = 0   # of the pair that positions turn least
        m[head - 2, 0] = w
        g.upload_f32_quantize(t, m.reshape(-1))
    g.finalize()
    prompt = np.array([huge] * 51 + [other] * 19 + [huge], dtype=np.int32)
    pos = len(prompt)
    _, _, logits = g.decode_sample_batch([prompt] + [prompt[-3:]] * 15, pos + 1, 0.0, 0.0, np.arange(1, 17), want_logits=True)
    for i, t in enumerate([1] + list(prompt)):
        want = g.forward(int(t), i)
        if i == 5:
            assert np.isnan(want).all()   # every row scores -inf
    assert np.isfinite(want).all()
    assert rel_err(logits[pos, 0], want) < 1e-4
    g.close()


@pytest.mark.parametrize("shape,n_seq,steps", [
    ((4096, 11008, 3, 32, 32, 32000, 48, 0), 32, 40),      # the widths of Llama-2-7B: rows of 16 and 43 groups
    ((4096, 11008, 3, 32, 32, 32000, 48, 0), 16, 40),
    ((8192, 28672, 2, 64, 8, 32000, 32, 0), 32, 24),       # the widths of Llama-2-70B: 64 heads on 8 kv heads, rows of 32 and 112 groups
])
def test_published_widths_match_the_single_decode_and_the_oracle(orc, shape, n_seq, steps):
    """At the matrix sizes of the published models (a few layers of them) every sequence of a batch gets the tokens of its
    own single-sequence decode, and four of them (the first, two in the middle, the one without a prompt) the oracle's
    tokens and, step by step, its logits."""
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(21, 0.02)
    g.finalize()
    rng = np.random.default_rng(n_seq + shape[0])
    prompts = [rng.integers(2, shape[5], size=int(rng.integers(0, 7))).astype(np.int32) for _ in range(n_seq - 1)]
    got, logits = g.decode_greedy_batch(prompts, steps, n_seq=n_seq, want_logits=True)
    for b in range(n_seq):
        p = prompts[b] if b < len(prompts) else np.zeros(0, dtype=np.int32)
        g.reset()
        want, _ = g.decode_greedy(p, steps)
        np.testing.assert_array_equal(got[b, :len(want)], want, err_msg="sequence %d" % b)
    g.close()
    m = oracle_of(orc, shape, 21)
    worst = 0.0
    for b in (0, n_seq // 3, n_seq // 2 + 1, n_seq - 1):
        p = prompts[b] if b < len(prompts) else np.zeros(0, dtype=np.int32)
        worst = max(worst, check_against_oracle(m, p, steps, got[b], logits[:, b], "sequence %d against the oracle" % b))
    print("batched logits vs oracle at widths %s: worst max|d|/max|logit| = %.3g" % (shape[:2], worst), flush=True)
    m.close()


def test_buffers_and_graph_are_kept_between_calls_and_replaced_when_they_do_not_fit():
    """The context owns the batched path's buffers: a second call with fewer steps and other prompts runs in them (other
    strides than its own arguments'), a call with more steps or another sequence count replaces them."""
    shape = (512, 1024, 2, 8, 2, 1008, 96, 0)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(5, 0.02)
    g.finalize()
    rng = np.random.default_rng(11)
    for n_seq, steps, longest in ((32, 48, 9), (32, 20, 4), (32, 64, 12), (16, 30, 6), (16, 30, 1)):
        prompts = [rng.integers(2, shape[5], size=int(rng.integers(0, longest + 1))).astype(np.int32) for _ in range(n_seq)]
        got, _ = g.decode_greedy_batch(prompts, steps, n_seq=n_seq)
        for b in (0, 1, n_seq - 1):
            g.reset()
            want, _ = g.decode_greedy(prompts[b], steps)
            np.testing.assert_array_equal(got[b, :len(want)], want, err_msg="%d sequences, %d steps, sequence %d" % (n_seq, steps, b))
    g.close()


def test_a_new_upload_replaces_the_tile_ordered_copy():
    """The batched products read a second copy of the matrices; uploading a tensor again must not leave the old copy in use."""
    shape = (512, 1024, 1, 8, 8, 1008, 16, 1)
    g = l2j.Transformer(l2j.Config(*shape))
    rng = np.random.default_rng(3)
    x = rng.standard_normal((16, 512)).astype(np.float32)
    for seed in (1, 2):
        g.fill_synthetic(seed, 0.02)      # (uploads are legal until finalize; the product does not need a finalized context)
        got, _ = g.batch_matmul(TENSOR.WQ, 0, x, 512)
        want = x.astype(np.float64) @ dequantized(g, TENSOR.WQ, 0, 512, 512).T
        assert (np.abs(got - want).max(axis=1) / np.abs(want).max(axis=1)).max() < 5e-6, seed
    g.close()


def test_shapes_the_batched_path_does_not_take_are_an_error():
    g = l2j.Transformer(l2j.Config(288, 768, 1, 6, 6, 320, 16, 1))   # rows of 288 codes: groups straddle rows
    g.fill_synthetic(1, 0.02)
    g.finalize()
    with pytest.raises(L2JError) as e:
        g.decode_greedy_batch([np.array([5, 6], dtype=np.int32)], 8)
    assert e.value.code == -2
    with pytest.raises(L2JError):
        g.batch_matmul(TENSOR.WQ, 0, np.zeros((16, 288), dtype=np.float32), 288)
    assert len(g.decode_greedy(np.array([5, 6], dtype=np.int32), 8)[0]) > 0     # the context stays usable
    g.close()


def test_sequence_counts_other_than_16_and_32_are_an_error():
    g = l2j.Transformer(l2j.Config(512, 1024, 1, 8, 8, 1008, 16, 1))
    g.fill_synthetic(1, 0.02)
    g.finalize()
    for n_seq in (1, 8, 17, 48, 64):
        with pytest.raises(L2JError) as e:
            g.decode_greedy_batch([np.array([5], dtype=np.int32)], 4, n_seq=n_seq)
        assert e.value.code == -1
    g.close()


@pytest.mark.parametrize("n_seq,t,topp,vocab", [(16, 0.9, 0.9, 1008), (32, 1.0, 1.0, 1008), (32, 1.3, 0.6, 1008), (32, 1.0, 0.9, 32000),
                                                (16, 0.7, 1.0, 32000)])
def test_sampled_batch_gives_every_sequence_its_own_sampler(orc, n_seq, t, topp, vocab):
    """l2j_decode_sample_batch: sequence b must get what the reference's loop with a Sampler(seed b) gives it (J/Run.java:623-685,
    J/Sampler.java).  The oracle's sampler is fed the batched path's own logits of every step (they agree with the oracle's
    forward pass to rounding only, and a draw within that of a step of the cumulative sum would part two correct runs):
    every token identical; and the logits of a step must be those of the tokens sampled before it, which the
    single-sequence forward pass, fed the sampled tokens, confirms."""
    from tests.test_gpu_parity import make_pair
    shape = SHAPES[0][:5] + (vocab,) + SHAPES[0][6:]    # (32000: a sampling step takes 125 compute units, two of them run side by side)
    m, g = make_pair(orc, shape, seed=17, realistic=True)
    rng = np.random.default_rng(n_seq)
    steps = 28 if vocab < 10000 else 14
    prompts = [rng.integers(3, vocab, size=int(rng.integers(0, 7))).astype(np.int32) for _ in range(n_seq - 2)]   # (two run without one)
    seeds = rng.integers(-2**40, 2**40, size=n_seq).astype(np.int64)
    got, sec, logits = g.decode_sample_batch(prompts, steps, t, topp, seeds, n_seq=n_seq, want_logits=True)
    assert got.shape == (n_seq, steps) and sec > 0
    for b in range(n_seq):
        prompt = prompts[b] if b < len(prompts) else np.zeros(0, dtype=np.int32)
        s = orc.Sampler(int(seeds[b]), vocab)
        want = [int(prompt[pos]) if pos < len(prompt) else s.step(logits[pos, b], t, topp)[0] for pos in range(steps)]
        np.testing.assert_array_equal(got[b], np.array(want, dtype=np.int32), err_msg="sequence %d" % b)
    for b in (0, n_seq - 1):                                     # the sampled tokens are what the next step reads
        g.reset()
        tok = 1
        for pos in range(steps):
            lg = g.forward(tok, pos)
            assert rel_err(logits[pos, b], lg.astype(np.float64)) < 1e-5, (b, pos)
            tok = int(got[b, pos])
    again, _ = g.decode_sample_batch(prompts, steps, t, topp, seeds, n_seq=n_seq)      # the seeds restart generators and arrays
    np.testing.assert_array_equal(again, got)
    other, _ = g.decode_sample_batch(prompts, steps, t, topp, seeds + 1, n_seq=n_seq)
    assert not np.array_equal(other, got)
    greedy, _ = g.decode_greedy_batch(prompts, steps, n_seq=n_seq)
    cold, _ = g.decode_sample_batch(prompts, steps, 0.0, topp, seeds, n_seq=n_seq)     # temperature 0: Sampler.argmax
    np.testing.assert_array_equal(cold, greedy)
    g.close()


@pytest.mark.parametrize("vocab,spread,least,most", [(272, 4.0, 1, 256), (1008, 20.0, 1, 256), (4112, 0.3, 4097, 4112), (8208, 3.0, 257, 4096),
                                                     (32000, 5.0, 1, 4096), (32000, 2.0, 8193, 20480), (36864, 1.0, 24577, 36864)])
def test_sampled_batch_merges_few_and_many_candidates_with_what_earlier_steps_left(orc, vocab, spread, least, most):
    """Top-p steps whose candidates are one tile (256 pairs), one run (4096), two, three to five or seven of the sort, by the logits' spread: every
    token the one that the oracle's sampler, which sorts its whole array, takes from the same logits."""
    shape = SHAPES[1][:5] + (vocab,) + SHAPES[1][6:]    # (a classifier of its own: with the embedding's a token's own logit stands out)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(23, 0.02)
    g.upload_f32_quantize(l2j.TENSOR.RMS_FINAL, np.full(shape[0], spread / (0.02 * shape[0] ** 0.5), dtype=np.float32))
    g.finalize()
    rng = np.random.default_rng(vocab)
    prompts = [rng.integers(3, vocab, size=int(rng.integers(0, 5))).astype(np.int32) for _ in range(16)]
    seeds = rng.integers(-2**40, 2**40, size=16).astype(np.int64)
    for t, topp in ((0.9, 0.9), (1.4, 0.5)):
        got, _, logits = g.decode_sample_batch(prompts, 12, t, topp, seeds, want_logits=True)
        for b in range(16):
            s = orc.Sampler(int(seeds[b]), vocab)
            want = [int(prompts[b][pos]) if pos < len(prompts[b]) else s.step(logits[pos, b], t, topp)[0] for pos in range(12)]
            np.testing.assert_array_equal(got[b], np.array(want, dtype=np.int32), err_msg="sequence %d" % b)
        p = np.exp((logits.astype(np.float64) - logits.max(axis=2, keepdims=True)) / t)
        n0 = (p / p.sum(axis=2, keepdims=True) >= (1 - topp) / (vocab - 1)).sum(axis=2)
        assert least <= n0.min() and n0.max() <= most, (t, int(n0.min()), int(n0.max()))
    g.close()


def test_sampled_batch_reports_what_the_sampler_reports_and_goes_on(orc):
    """A NaN in the logits of one sequence, and a flat distribution with topp 0, which leaves no candidate: both an error, from top-p and (the NaN)
    plain sampling, and the next call of the same context gives every sequence the oracle's tokens."""
    shape = SHAPES[1]
    vocab, dim, n_seq, steps = shape[5], shape[0], 16, 10
    rng = np.random.default_rng(8)
    emb = (0.02 * rng.standard_normal((vocab, dim))).astype(np.float32)
    emb[5, 7] = np.nan
    prompts = [rng.integers(6, vocab, size=b % 4).astype(np.int32) for b in range(n_seq)]
    bad = [np.array([9, 5], dtype=np.int32) if b == 11 else p for b, p in enumerate(prompts)]
    seeds = np.arange(n_seq) + 70

    def check(g, t, topp):
        got, _, logits = g.decode_sample_batch(prompts, steps, t, topp, seeds, want_logits=True)
        for b in range(n_seq):
            s = orc.Sampler(int(seeds[b]), vocab)
            want = [int(prompts[b][pos]) if pos < len(prompts[b]) else s.step(logits[pos, b], t, topp)[0] for pos in range(steps)]
            want = np.array(want, dtype=np.int32)
            if 5 not in want:                                            # (else the sequence has drawn the NaN itself)
                np.testing.assert_array_equal(got[b], want, err_msg="sequence %d" % b)

    for spread in (4.0, 0.0):
        g = l2j.Transformer(l2j.Config(*shape))
        g.fill_synthetic(23, 0.02)
        g.upload_f32(TENSOR.TOK_EMB, emb)
        g.upload_f32_quantize(TENSOR.RMS_FINAL, np.full(dim, spread / (0.02 * dim ** 0.5), dtype=np.float32))
        g.finalize()
        if spread:
            for topp in (0.9, 1.0):
                with pytest.raises(L2JError, match="NaN"):
                    g.decode_sample_batch(bad, steps, 0.9, topp, seeds)
                check(g, 0.5, topp)
        else:
            with pytest.raises(L2JError, match="cutoff"):
                g.decode_sample_batch(prompts, steps, 1.0, 0.0, seeds)
            check(g, 1.0, 0.9)
        g.close()


def test_sampled_batch_refuses_what_its_sampling_step_cannot_take():
    g = l2j.Transformer(l2j.Config(*SHAPES[3]))
    g.fill_synthetic(3, 0.02)
    g.finalize()
    p = [np.array([5, 6], dtype=np.int32)]
    with pytest.raises(L2JError):
        g.decode_sample_batch(p, 8, -1.0, 0.9, [1])
    with pytest.raises(L2JError):
        g.decode_sample_batch(p, 8, 1.0, 1.5, [1])
    g.set_option("sampler_scan", 0)
    with pytest.raises(L2JError, match="sampler_scan"):
        g.decode_sample_batch(p, 8, 1.0, 0.9, [1])
    g.set_option("sampler_scan", 1)
    g.set_option("sampler_wide", 0)                      # (the one-launch step of the single sequence: not what the batch takes)
    out, _ = g.decode_sample_batch(p, 8, 1.0, 0.9, [1])
    assert out.shape == (16, 8) and np.array_equal(out[0, :2], p[0])
    g.close()


def test_the_sampling_steps_of_the_batch_wait_for_nobody():
    """barrier_spins 0 makes every bounded wait between workgroups give up at once; the batch's sampling steps have none (a
    launch per stage, the sequences side by side in each): the tokens of a context with the default."""
    shape = SHAPES[0]
    outs = []
    for spins in (None, 0):
        g = l2j.Transformer(l2j.Config(*shape))
        g.fill_synthetic(5, 0.02)
        if spins is not None:
            g.set_option("barrier_spins", spins)
        g.finalize()
        out, _ = g.decode_sample_batch([np.array([9, 8, 7], dtype=np.int32)], 12, 1.0, 0.9, [3])
        outs.append(out)
        g.close()
    np.testing.assert_array_equal(outs[0], outs[1])


def test_release_batch_gives_the_memory_back_and_the_next_call_makes_it_again():
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = C.c_size_t(0), C.c_size_t(0)
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    shape = SHAPES[2]
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(11, 0.02)
    g.finalize()
    prompts = [np.array([5, 9, 13], dtype=np.int32), np.array([7], dtype=np.int32)]
    single, _ = g.decode_greedy(prompts[0], 24)
    g.reset()
    g.release_batch()                                  # (nothing to release yet: not an error)
    before = free_bytes()
    want, _ = g.decode_greedy_batch(prompts, 24)
    sampled, _ = g.decode_sample_batch(prompts, 24, 0.9, 0.9, [1, 2])
    tokens = np.concatenate([[1], prompts[0], np.arange(20, 40)]).astype(np.int32)
    logits, _ = g.prefill(tokens)
    held = before - free_bytes()
    assert held > 10 << 20                             # the copy of the matrices, caches, buffers, samplers
    g.release_batch()
    assert abs(free_bytes() - before) <= 4 << 20
    g.reset()
    again, _ = g.decode_greedy_batch(prompts, 24)
    np.testing.assert_array_equal(again, want)
    np.testing.assert_array_equal(g.decode_sample_batch(prompts, 24, 0.9, 0.9, [1, 2])[0], sampled)
    g.reset()
    np.testing.assert_array_equal(g.prefill(tokens)[0].view(np.uint32), logits.view(np.uint32))
    g.reset()
    np.testing.assert_array_equal(g.decode_greedy(prompts[0], 24)[0], single)   # the single-sequence path: untouched
    g.close()


@pytest.mark.parametrize("n_seq,shortest,longest", [(16, 1, 1), (16, 2, 5), (32, 15, 18), (32, 33, 40), (16, 66, 70)])
def test_common_prompt_positions_taken_at_once(orc, n_seq, shortest, longest):
    """Prompts for every sequence: the positions whose inputs all sequences know (up to the shortest prompt) are one pass, or
    several (1024 rows each), the loop goes on behind them.  Tokens as every sequence decodes alone, with and without the
    logits kept, and the logits of every step the oracle's."""
    shape = SHAPES[1][:6] + (80,) + SHAPES[1][7:]
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(n_seq + shortest)
    lengths = rng.integers(shortest, longest + 1, size=n_seq)
    lengths[1], lengths[2] = shortest, longest
    prompts = [rng.integers(2, shape[5], size=int(n)).astype(np.int32) for n in lengths]
    for steps in (longest + 6, max(1, shortest - 1)):        # on behind the prompts; inside them
        got, sec = g.decode_greedy_batch(prompts, steps, n_seq=n_seq)
        assert sec >= 0
        kept, logits = g.decode_greedy_batch(prompts, steps, n_seq=n_seq, want_logits=True)
        np.testing.assert_array_equal(kept, got)
        m = oracle_of(orc, shape, 9)
        for b in range(n_seq):
            g.reset()
            want, _ = g.decode_greedy(prompts[b], steps)
            same_until_a_tie(got[b, :len(want)], want, logits[:, b], "sequence %d" % b)
            if b < 4:
                check_against_oracle(m, prompts[b], steps, got[b], logits[:, b], "sequence %d against the oracle" % b)
        m.close()
        seeds = rng.integers(0, 2**40, size=n_seq).astype(np.int64)
        sampled, _, lg = g.decode_sample_batch(prompts, steps, 0.9, 0.9, seeds, n_seq=n_seq, want_logits=True)
        again, _ = g.decode_sample_batch(prompts, steps, 0.9, 0.9, seeds, n_seq=n_seq)
        np.testing.assert_array_equal(again, sampled)
        for b in (0, 1, 2, n_seq - 1):
            s = orc.Sampler(int(seeds[b]), shape[5])
            want = [int(prompts[b][pos]) if pos < lengths[b] else s.step(lg[pos, b], 0.9, 0.9)[0] for pos in range(steps)]
            np.testing.assert_array_equal(sampled[b], np.array(want, dtype=np.int32), err_msg="sequence %d" % b)
    g.close()


@pytest.mark.parametrize("n_seq", [16, 32])
def test_a_sequence_that_is_not_finite_leaves_earlier_positions_and_the_others_alone(n_seq):
    """A token whose embedding holds a NaN inside the common prompt: the logits of every other sequence, and of the positions before
    it of its own, are the bits they are with another token there."""
    shape = SHAPES[1]
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    rng = np.random.default_rng(n_seq)
    emb = (0.02 * rng.standard_normal((shape[5], shape[0]))).astype(np.float32)
    emb[5, 3] = np.nan
    g.upload_f32(TENSOR.TOK_EMB, emb)
    g.finalize()
    prompts = [rng.integers(6, shape[5], size=24).astype(np.int32) for _ in range(n_seq)]
    _, want = g.decode_greedy_batch(prompts, 25, n_seq=n_seq, want_logits=True)
    bad = [p.copy() for p in prompts]
    bad[3][9] = 5                                         # the input of position 10
    _, got = g.decode_greedy_batch(bad, 25, n_seq=n_seq, want_logits=True)
    others = [b for b in range(n_seq) if b != 3]
    np.testing.assert_array_equal(got[:, others].view(np.uint32), want[:, others].view(np.uint32))
    np.testing.assert_array_equal(got[:10, 3].view(np.uint32), want[:10, 3].view(np.uint32))
    assert np.isnan(got[10:, 3]).all()
    g.close()


@pytest.mark.parametrize("shape,tensor,rows,K", [
    ((1024, 2816, 2, 8, 4, 2000, 96, 0), "W1", 2816, 1024),   # rows in pairs of tiles: k_dstream
    ((1024, 2816, 2, 8, 4, 2000, 96, 0), "W2", 1024, 2816),
    ((768, 512, 2, 48, 3, 512, 40, 0), "WK", 48, 768),        # an odd number of tiles: k_dgemm
])
def test_a_product_keeps_its_precision_at_every_magnitude(shape, tensor, rows, K):
    """Activations from 2^-120 to 2^110, and with outliers a hundred times larger within a group: the relative error
    (2-norm over the outputs of a vector) stays below 3e-7 (1.0e-7 to 1.5e-7 measured; three bf16 planes per activation, before the
    digits, had 3.3e-7 to 5.0e-7)."""
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(7, 0.02)
    g.finalize()
    tensor = getattr(TENSOR, tensor)
    W = dequantized(g, tensor, 1, rows, K)
    rng = np.random.default_rng(K)
    normal = rng.standard_normal((16, K))
    outliers = normal * np.where(rng.random((16, K)) < 0.004, 100.0, 1.0)
    spread = np.ldexp(normal, rng.integers(-120, 20, (16, K // 256)).repeat(256, axis=1))     # every group of every vector another magnitude
    apart = np.ldexp(normal, rng.integers(-60, 110, (16, 1)))                                 # every vector another one
    for what, x in [("outliers", outliers), ("spread", spread), ("apart", apart)] + [("2^%d" % p, np.ldexp(normal, p)) for p in (110, 60, 0, -60, -90, -100, -110, -120)]:
        x = x.astype(np.float32)
        want = x.astype(np.float64) @ W.T
        got, _ = g.batch_matmul(tensor, 1, x, rows)
        err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() < 3e-7, (what, float(err.max()))
    zero, _ = g.batch_matmul(tensor, 1, np.zeros((16, K), dtype=np.float32), rows)
    assert not zero.any()
    g.close()


def test_a_product_keeps_its_precision_where_scales_are_small():
    """k_dgemm where a vector's 2^-s times a row's scale lies below 2^-126, and no sums are kept times 2^48: a matrix of 2^-68, and vectors of
    2^-95 that share a tile with one of 2^60.  The bound of the other magnitudes."""
    shape, rows, K = (768, 512, 1, 48, 3, 512, 40, 0), 48, 768
    rng = np.random.default_rng(1)
    normal = rng.standard_normal((16, K))
    w = 0.02 * rng.standard_normal((rows, K))
    for power, x in ((-62, np.ldexp(normal, -33)), (0, np.ldexp(normal, np.array([60] + [-95] * 15)[:, None]))):
        g = l2j.Transformer(l2j.Config(*shape))
        g.upload_f32_quantize(TENSOR.WK, np.ldexp(w, power))
        W = dequantized(g, TENSOR.WK, 0, rows, K)
        x = x.astype(np.float32)
        want = x.astype(np.float64) @ W.T
        got, _ = g.batch_matmul(TENSOR.WK, 0, x, rows)
        g.close()
        err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() < 3e-7, (power, float(err.max()))


class FullDevice:
    """All of the device's free memory but `leave` bytes, held for the duration of a with block."""

    def __init__(self, leave):
        import ctypes as C
        self.C, self.hip, self.leave, self.held = C, C.CDLL("libamdhip64.so"), leave, []

    def free_bytes(self):
        free, total = self.C.c_size_t(0), self.C.c_size_t(0)
        assert self.hip.hipMemGetInfo(self.C.byref(free), self.C.byref(total)) == 0
        return free.value

    def __enter__(self):
        while self.free_bytes() > self.leave + (4 << 20):
            p = self.C.c_void_p()
            n = min(self.free_bytes() - self.leave, 32 << 30) & ~((2 << 20) - 1)
            assert self.hip.hipMalloc(self.C.byref(p), self.C.c_size_t(n)) == 0
            self.held.append(p)
        return self

    def __exit__(self, *a):
        for p in self.held:
            self.hip.hipFree(p)


def test_known_positions_go_through_the_loop_where_the_memory_for_their_pass_is_missing():
    """The pass over the known prompt positions is a shortcut: with room for half its rows it runs in smaller passes, with room for
    none the loop takes every position.  The tokens are those of the run with all the memory."""
    shape = (256, 28672, 1, 1, 1, 512, 64, 1)         # a row's hidden products are large: 205 MB for the step's 32 rows, 630 for 672
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(5)
    prompts = [rng.integers(2, shape[5], size=20).astype(np.int32) for _ in range(32)]
    want, logits = g.decode_greedy_batch(prompts, 30, n_seq=32, want_logits=True)
    for leave in (420 << 20, 120 << 20):
        g.release_batch()
        g.decode_greedy_batch([p[:0] for p in prompts[:31]] + [prompts[31]], 30, n_seq=32)     # the step's buffers, prompts of this length
        with FullDevice(leave):
            got, _ = g.decode_greedy_batch(prompts, 30, n_seq=32)
        for b in range(32):
            same_until_a_tie(got[b], want[b], logits[:, b], "sequence %d, %d MB" % (b, leave >> 20))
    g.close()


def test_the_logits_of_every_step_come_through_as_many_slots_as_there_is_memory_for():
    """65 MB of logits per step (a vocabulary of 512000, 32 sequences): all slots, a few, one; and a short call keeps no more than it
    has steps.  The same logits to the bit."""
    shape = (256, 256, 1, 1, 1, 512000, 64, 1)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    prompts = [np.array([7 + b, 9], dtype=np.int32) for b in range(32)]
    want_tokens, want = g.decode_greedy_batch(prompts, 9, n_seq=32, want_logits=True)
    for leave in (320 << 20, 100 << 20):
        g.release_batch()
        g.decode_greedy_batch(prompts, 9, n_seq=32)                  # the step's buffers
        with FullDevice(leave) as full:
            got_tokens, got = g.decode_greedy_batch(prompts, 9, n_seq=32, want_logits=True)
            assert full.free_bytes() < leave - (60 << 20)
        np.testing.assert_array_equal(got_tokens, want_tokens)
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    g.release_batch()
    g.decode_greedy_batch(prompts, 2, n_seq=32)
    before = FullDevice(0).free_bytes()
    g.decode_greedy_batch(prompts, 2, n_seq=32, want_logits=True)
    assert before - FullDevice(0).free_bytes() < 3 * 66 << 20        # two slots of 65 MB
    g.close()


def test_a_call_after_one_that_found_no_memory_is_not_blamed_for_it():
    """The error of a failed allocation stays behind in the runtime: the calls that follow a failed one, of its context and of
    others, must not take it for their own launches'."""
    shape = (256, 28672, 1, 1, 1, 512, 64, 1)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    prompt = np.array([5, 6, 7], dtype=np.int32)
    want, _ = g.decode_greedy(prompt, 24)
    with FullDevice(100 << 20):
        with pytest.raises(L2JError, match="out of memory"):
            g.decode_greedy_batch([prompt], 24, n_seq=32)
        g.reset()
        np.testing.assert_array_equal(g.decode_greedy(prompt, 24)[0], want)
        with pytest.raises(L2JError, match="out of memory"):
            l2j.Transformer(l2j.Config(4096, 11008, 4, 32, 32, 512, 64, 0))
        g.forward(1, 0)
    np.testing.assert_array_equal(g.decode_greedy_batch([prompt], 24, n_seq=32)[0][0, :len(want)], want)
    g.close()


@pytest.mark.parametrize("heads,kv_heads", [(64, 8), (32, 32), (16, 4)])       # head 64, 128, 256
@pytest.mark.parametrize("n_seq,shortest", [(16, 19), (16, 40), (16, 70), (32, 16), (32, 40)])
def test_common_prompt_positions_of_a_wide_model(heads, kv_heads, n_seq, shortest):
    """4096 wide, the attention of a pass has a workgroup for two blocks of a sequence: 20 positions of 16 sequences are two blocks of
    16, 41 two of 32 (three of 16 with head size 256), 71 two passes.  The logits of every step and sequence against l2j_forward
    on the sequence's tokens."""
    shape = (4096, 1024, 2, heads, kv_heads, 512, 96, 0)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(heads + shortest)
    prompts = [rng.integers(2, shape[5], size=shortest + int(rng.integers(0, 3))).astype(np.int32) for _ in range(n_seq)]
    prompts[n_seq - 1] = prompts[n_seq - 1][:shortest]
    steps = shortest + 4
    tokens, logits = g.decode_greedy_batch(prompts, steps, n_seq=n_seq, want_logits=True)
    for b in range(0, n_seq, 1 if n_seq == 16 else 3):
        g.reset()
        for pos in range(steps):
            want = g.forward(1 if pos == 0 else int(tokens[b, pos - 1]), pos)
            assert rel_err(logits[pos, b], want.astype(np.float64)) < 2e-5, (b, pos)
            assert tokens[b, pos] == (prompts[b][pos] if pos < len(prompts[b]) else np.argmax(logits[pos, b])), (b, pos)
    g.close()


def test_a_longer_common_prompt_allocates_nothing_where_the_prompts_fit():
    """The first call whose prompts all have ids makes room for the longest common prompt its buffers take."""
    shape = (512, 8192, 1, 8, 8, 512, 96, 1)              # (64 positions of 16 sequences: 270 MB)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(9, 0.02)
    g.finalize()
    rng = np.random.default_rng(8)
    full = [rng.integers(2, shape[5], size=70).astype(np.int32) for _ in range(16)]
    g.decode_greedy_batch([full[0]] + [p[:2] for p in full[1:]], 80, n_seq=16)
    before = FullDevice(0).free_bytes()
    for shortest in (9, 30, 70):
        g.decode_greedy_batch([full[0]] + [p[:shortest] for p in full[1:]], 80, n_seq=16)
        assert FullDevice(0).free_bytes() == before, shortest
    g.close()
