"""l2j_prefill: the prompt positions of the token loop (J/Run.java:623-640, one Run.transformer call per position in the
reference) many at once through the batched products.  It must leave in the KV cache, and return for the last position,
what l2j_forward position by position does (to rounding: the sums are formed in another order), and both must be what the
CPU oracle computes."""
import numpy as np
import pytest

import llama2j_amd as l2j
from llama2j_amd.binding import BUFFER, TENSOR, L2JError
from tests.test_gpu_batch import FullDevice, LOGIT_TOL, dequantized, oracle_of, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [
    (512, 1024, 4, 8, 8, 1008, 80, 1),      # head 64, shared classifier
    (512, 1024, 2, 8, 2, 1008, 72, 0),      # grouped-query attention: 8 heads on 2 kv heads
    (1024, 2816, 2, 8, 4, 2000, 96, 0),     # head 128, an odd number of groups per row
    (512, 768, 2, 2, 2, 512, 40, 1),        # head 256
]
CLOSE = 2e-5   # prefill against l2j_forward: relative to the largest value of what is compared


def model(shape, seed=9):
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(seed, 0.02)
    g.finalize()
    return g


def caches(g, shape):
    return [np.stack([g.read(which, layer) for layer in range(shape[2])]) for which in (BUFFER.KCACHE, BUFFER.VCACHE)]


@pytest.mark.parametrize("flash", [2, 0])    # the keys of 16 positions shared by the waves of a workgroup: always / never (default: few positions behind 512 keys or more)
@pytest.mark.parametrize("shape", SHAPES)
def test_prefill_leaves_what_forward_position_by_position_leaves(orc, shape, flash):
    seq_len, kvd = shape[6], shape[0] // shape[3] * shape[4]
    rng = np.random.default_rng(shape[0] + shape[6])
    g = model(shape)
    g.set_option("prefill_flash", flash)
    m = oracle_of(orc, shape, 9)
    for n in (1, 31, 32, 33, seq_len):
        tokens = np.concatenate([[1], rng.integers(2, shape[5], size=n - 1)]).astype(np.int32)   # BOS first (J/Run.java:612)
        g.reset()
        for i, t in enumerate(tokens):
            want_logits = g.forward(int(t), i)
        want_k, want_v = caches(g, shape)
        g.reset()
        got_logits, sec = g.prefill(tokens)
        got_k, got_v = caches(g, shape)
        assert sec > 0
        assert rel_err(got_logits, want_logits.astype(np.float64)) < CLOSE, n
        for got, want in ((got_k, want_k), (got_v, want_v)):
            got, want = got.reshape(shape[2], seq_len, kvd), want.reshape(shape[2], seq_len, kvd)
            assert rel_err(got[:, :n], want[:, :n].astype(np.float64)) < CLOSE, n
            assert not got[:, n:].any(), n                      # rows past the last position: untouched
        # and the oracle, from the same tokens: the logits of the last position within the bar
        m.reset()
        for i, t in enumerate(tokens):
            oracle_logits = m.forward(int(t), i)
        assert rel_err(got_logits, oracle_logits.astype(np.float64)) < LOGIT_TOL, n
    m.close()


@pytest.mark.parametrize("n", [1, 2, 17, 65, 511, 513, 1030])   # ... up to where the last position's attention changes kernels, and two passes
@pytest.mark.parametrize("shape", [(512, 768, 1, 8, 2, 512, 1040, 0), (512, 1024, 1, 2, 2, 512, 1040, 1)])
def test_the_last_layer_for_the_last_position_alone(shape, n):
    # one layer: all that is behind its keys and values is for one row
    tokens = np.random.default_rng(n).integers(2, shape[5], size=n).astype(np.int32)
    g = model(shape)
    got, _ = g.prefill(tokens)
    k, v = caches(g, shape)
    after = g.forward(3, n)
    g.reset()
    for i, t in enumerate(tokens):
        want = g.forward(int(t), i)
    assert rel_err(got, want.astype(np.float64)) < CLOSE
    for a, b in zip((k, v), caches(g, shape)):
        assert rel_err(a, b.astype(np.float64)) < CLOSE
    assert rel_err(after, g.forward(3, n).astype(np.float64)) < CLOSE
    g.close()


@pytest.mark.parametrize("n", [2, 15, 16, 17, 31, 32])
def test_swiglu_within_the_products_with_vectors_missing(n):
    # up to 16 and up to 32 vectors, whole and not
    shape = (1024, 2048, 2, 8, 8, 512, 40, 1)
    tokens = np.random.default_rng(n).integers(2, shape[5], size=n).astype(np.int32)
    g = model(shape)
    got, _ = g.prefill(tokens)
    for i, t in enumerate(tokens):
        want = g.forward(int(t), i)
    assert rel_err(got, want.astype(np.float64)) < CLOSE
    g.close()
    # an activation that is not finite: its group's scale is a NaN, and no other vector's
    test_values_that_are_not_finite_stay_behind_the_causal_mask((512, 1024, 2, 8, 2, 1008, 64, 0), max(n, 12), 1, 0)


@pytest.mark.parametrize("shape", SHAPES[:2])
def test_prefill_goes_on_from_a_position_and_decode_goes_on_from_prefill(orc, shape):
    seq_len = shape[6]
    rng = np.random.default_rng(shape[6])
    g = model(shape)
    n1, n2, more = 17, 40, 8
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=n1 + n2 - 1)]).astype(np.int32)
    g.reset()
    whole, _ = g.prefill(tokens)
    k_whole, v_whole = caches(g, shape)
    g.reset()
    g.prefill(tokens[:n1], want_logits=False)
    parts, _ = g.prefill(tokens[n1:], pos0=n1)
    k_parts, v_parts = caches(g, shape)
    assert rel_err(parts, whole.astype(np.float64)) < CLOSE
    assert rel_err(k_parts, k_whole.astype(np.float64)) < CLOSE and rel_err(v_parts, v_whole.astype(np.float64)) < CLOSE
    # the single-sequence path continues on the cache prefill has left: the logits of the next positions against a run
    # that took every position through l2j_forward
    nxt = rng.integers(2, shape[5], size=more).astype(np.int32)
    after_prefill = [g.forward(int(t), n1 + n2 + i) for i, t in enumerate(nxt)]
    g.reset()
    for i, t in enumerate(np.concatenate([tokens, nxt])):
        lg = g.forward(int(t), i)
        if i >= n1 + n2:
            assert rel_err(after_prefill[i - n1 - n2], lg.astype(np.float64)) < CLOSE, i
    assert n1 + n2 + more <= seq_len


def test_prefill_refuses_what_it_cannot_take(orc):
    g = model(SHAPES[0])
    with pytest.raises(L2JError):
        g.prefill(np.array([1, 5000], dtype=np.int32))          # token id beyond the vocabulary
    with pytest.raises(L2JError):
        g.prefill(np.ones(4, dtype=np.int32), pos0=SHAPES[0][6] - 2)   # past seq_len
    small = l2j.Transformer(l2j.Config(64, 128, 2, 4, 4, 512, 32, 1))       # dim not in whole groups of 256
    small.fill_synthetic(3, 0.1)
    small.finalize()
    with pytest.raises(L2JError):
        small.prefill(np.array([1, 2, 3], dtype=np.int32))


@pytest.mark.parametrize("shape,n_prompt", [(SHAPES[0], 40), (SHAPES[1], 65), (SHAPES[2], 33)])
def test_decode_loops_with_option_prefill_give_the_tokens_they_give_without(orc, shape, n_prompt):
    """Option prefill: the loops take a prompt of eight ids or more through l2j_prefill and go on from there.
    Greedy against the CPU oracle's loop as well; sampled with the same seed."""
    steps = shape[6]
    prompt = orc.synth_prompt(5, n_prompt, shape[5])
    g = model(shape)
    want, _ = g.decode_greedy(prompt, steps)
    want_s, _ = g.decode_sample(prompt, steps, 0.9, 0.9, 11)
    g.set_option("prefill", 1)
    g.reset()
    got, sec = g.decode_greedy(prompt, steps)
    assert sec > 0
    np.testing.assert_array_equal(got, want)
    g.reset()
    got_s, _ = g.decode_sample(prompt, steps, 0.9, 0.9, 11)
    np.testing.assert_array_equal(got_s, want_s)
    m = oracle_of(orc, shape, 9)
    cpu, _, _ = m.generate_greedy(prompt, steps)
    np.testing.assert_array_equal(got[:len(cpu)], cpu)
    m.close()
    # a prompt id 1 ends the loop there, as without the option
    stop = prompt.copy()
    stop[7] = 1
    g.reset()
    got, _ = g.decode_greedy(stop, steps)
    assert len(got) == 8 and got[-1] == 1


@pytest.mark.parametrize("shape,n", [
    ((4096, 11008, 3, 32, 32, 32000, 48, 0), 45),      # the widths of Llama-2-7B (three layers of it)
    ((8192, 28672, 2, 64, 8, 32000, 40, 0), 37),       # the widths of Llama-2-70B: 64 heads on 8 kv heads
])
def test_prefill_at_the_published_widths(orc, shape, n):
    rng = np.random.default_rng(n)
    g = l2j.Transformer(l2j.Config(*shape))
    g.fill_synthetic(21, 0.02)
    g.finalize()
    g.set_option("prefill_flash", 2)
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=n - 1)]).astype(np.int32)
    for i, t in enumerate(tokens):
        want = g.forward(int(t), i)
    g.reset()
    got, _ = g.prefill(tokens)
    assert rel_err(got, want.astype(np.float64)) < CLOSE
    g.close()
    m = oracle_of(orc, shape, 21)
    for i, t in enumerate(tokens):
        cpu = m.forward(int(t), i)
    worst = rel_err(got, cpu.astype(np.float64))
    print("prefill logits vs oracle at widths %s: max|d|/max|logit| = %.3g" % (shape[:2], worst), flush=True)
    assert worst < LOGIT_TOL
    m.close()


def test_prefill_and_the_batched_decode_share_their_buffers(orc):
    """Both use the context's copy of the matrices, and the prompts of a batch run in prefill's buffers: calls of either kind in any
    order give what they give alone."""
    shape = SHAPES[1]
    g = model(shape)
    rng = np.random.default_rng(3)
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=44)]).astype(np.int32)
    prompts = [rng.integers(2, shape[5], size=3).astype(np.int32) for _ in range(16)]
    alone_logits, _ = g.prefill(tokens)
    alone_tokens, _ = g.decode_greedy_batch(prompts, 24, n_seq=16)        # (its prompts' pass in prefill's buffers)
    g.reset()
    again_logits, _ = g.prefill(tokens)
    assert np.array_equal(again_logits.view(np.uint32), alone_logits.view(np.uint32))
    again_tokens, _ = g.decode_greedy_batch(prompts + prompts, 24, n_seq=32)
    np.testing.assert_array_equal(again_tokens[:16], alone_tokens)
    g.reset()
    third, _ = g.prefill(tokens)                                          # (in the buffers the 32 sequences' pass has grown)
    assert np.array_equal(third.view(np.uint32), alone_logits.view(np.uint32))


def test_prefill_past_the_position_where_the_attention_changes_kernels(orc):
    """By default a pass of few positions over 512 keys or more shares the keys of 16 positions among the waves of a workgroup, and
    among up to four workgroups: 470 positions at once stay below; behind 480 cached ones 16, 40 and 100 positions have four
    workgroups per head and block, 180 two, 300 one.  Against position-by-position forwards and the oracle."""
    shape = (512, 1024, 2, 8, 2, 1008, 800, 0)
    kvd = 512 * 2 // 8
    rng = np.random.default_rng(640)
    g = model(shape)
    n = 470
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=n - 1)]).astype(np.int32)
    for i, t in enumerate(tokens):
        want = g.forward(int(t), i)
    want_k, want_v = caches(g, shape)
    g.reset()
    got, _ = g.prefill(tokens)
    got_k, got_v = caches(g, shape)
    assert rel_err(got, want.astype(np.float64)) < CLOSE
    assert rel_err(got_k, want_k.astype(np.float64)) < CLOSE and rel_err(got_v, want_v.astype(np.float64)) < CLOSE
    m = oracle_of(orc, shape, 9)
    for i, t in enumerate(tokens):
        cpu = m.forward(int(t), i)
    assert rel_err(got, cpu.astype(np.float64)) < LOGIT_TOL
    cached, behind = 480, (16, 40, 100, 180, 300)
    tokens = np.concatenate([tokens, rng.integers(2, shape[5], size=cached + max(behind) - n)]).astype(np.int32)
    wants = {}
    g.reset()
    for i, t in enumerate(tokens):
        lg = g.forward(int(t), i)
        if i + 1 - cached in behind:
            wants[i + 1 - cached] = lg
    want_k, want_v = (x.reshape(shape[2], shape[6], kvd) for x in caches(g, shape))
    for more in behind:
        end = cached + more
        g.reset()
        g.prefill(tokens[:cached], want_logits=False)
        got, _ = g.prefill(tokens[cached:end], pos0=cached)
        got_k, got_v = (x.reshape(shape[2], shape[6], kvd) for x in caches(g, shape))
        assert rel_err(got, wants[more].astype(np.float64)) < CLOSE, more
        assert rel_err(got_k[:, :end], want_k[:, :end].astype(np.float64)) < CLOSE and rel_err(got_v[:, :end], want_v[:, :end].astype(np.float64)) < CLOSE, more
    for i in range(n, len(tokens)):
        cpu = m.forward(int(tokens[i]), i)
    assert rel_err(got, cpu.astype(np.float64)) < LOGIT_TOL
    m.close()


@pytest.mark.parametrize("shape", SHAPES)
def test_the_keys_of_a_head_split_over_one_to_four_workgroups(shape):
    """Option prefill_split: as many workgroups share the keys of a head in the matrix-core attention, the last of them to finish
    merging what the others left (also where there are fewer tiles of 16 keys than workgroups): the logits and cache rows of
    position-by-position forwards, for every head size, and twice in a row (the counters of a launch are left at zero)."""
    seq_len = shape[6]
    rng = np.random.default_rng(seq_len)
    g = model(shape)
    g.set_option("prefill_flash", 2)
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=seq_len - 1)]).astype(np.int32)
    for i, t in enumerate(tokens):
        want = g.forward(int(t), i)
    want_k, want_v = caches(g, shape)
    for split in (4, 3, 2, 1, 4):
        g.set_option("prefill_split", split)
        g.reset()
        got, _ = g.prefill(tokens)
        got_k, got_v = caches(g, shape)
        assert rel_err(got, want.astype(np.float64)) < CLOSE, split
        assert rel_err(got_k, want_k.astype(np.float64)) < CLOSE and rel_err(got_v, want_v.astype(np.float64)) < CLOSE, split
    g.close()


@pytest.mark.parametrize("shape", [
    (512, 1024, 2, 8, 2, 1008, 1104, 0),     # head 64, grouped-query attention: a wave per 16 positions and shared keys
    (256, 768, 2, 1, 1, 512, 304, 1),        # head 256, one head: one group per row, three per hidden row
])
def test_passes_of_many_positions(shape):
    """Edges of the tiles of 32 and 64 positions, of a pass (1024 positions; one more makes two passes of half), and a second
    call behind cached positions, against position by position: logits of the last position and the cache rows."""
    seq_len, kvd = shape[6], shape[0] // shape[3] * shape[4]
    rng = np.random.default_rng(shape[0])
    g = model(shape)
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=seq_len - 1)]).astype(np.int32)
    sizes = [n for n in (2, 63, 64, 65, 129, 255, 256, 257, 300, 1024, 1025, 1104) if n <= seq_len]
    want = {}
    for i, t in enumerate(tokens):
        lg = g.forward(int(t), i, want_logits=i + 1 in sizes)
        if i + 1 in sizes:
            want[i + 1] = lg
    want_k, want_v = (x.reshape(shape[2], seq_len, kvd) for x in caches(g, shape))
    for n in sizes:
        for first in ((0,) if n < 65 else (0, n // 3)):
            g.reset()
            if first:
                g.prefill(tokens[:first], want_logits=False)
            got, _ = g.prefill(tokens[first:n], pos0=first)
            assert rel_err(got, want[n].astype(np.float64)) < CLOSE, (n, first)
            k, v = (x.reshape(shape[2], seq_len, kvd) for x in caches(g, shape))
            assert rel_err(k[:, :n], want_k[:, :n].astype(np.float64)) < CLOSE, (n, first)
            assert rel_err(v[:, :n], want_v[:, :n].astype(np.float64)) < CLOSE, (n, first)
            assert not k[:, n:].any() and not v[:, n:].any(), (n, first)
    g.close()


@pytest.mark.parametrize("shape,n,flash,split", [
    ((512, 1024, 2, 8, 2, 1008, 64, 0), 40, 1, 0),        # head 64: blocks of 16 positions
    ((4096, 512, 2, 32, 8, 512, 608, 0), 600, 1, 0),      # head 128: pairs of blocks of 32
    ((4096, 512, 2, 16, 16, 512, 304, 0), 300, 1, 0),     # head 256: pairs of blocks of 16
    ((512, 1024, 2, 8, 2, 1008, 64, 0), 40, 2, 1),        # the keys shared by the waves of a workgroup,
    ((1024, 512, 2, 8, 4, 512, 64, 0), 50, 2, 4),         # and by four workgroups
    ((512, 768, 2, 2, 2, 512, 40, 1), 38, 2, 1),
])
def test_values_that_are_not_finite_stay_behind_the_causal_mask(shape, n, flash, split):
    """A token whose embedding holds a NaN, in the middle of a tile of keys: the positions before it attend to none of its
    rows and keep theirs, to the bit, and all positions from it on are NaN from the second layer's rows on."""
    kvd = shape[0] // shape[3] * shape[4]
    rng = np.random.default_rng(n)
    g = l2j.Transformer(l2j.Config(*shape), options={"prefill_flash": flash, "prefill_split": split})
    g.fill_synthetic(9, 0.02)
    emb = (0.02 * rng.standard_normal((shape[5], shape[0]))).astype(np.float32)
    emb[5, 3] = np.nan
    g.upload_f32(TENSOR.TOK_EMB, emb)
    g.finalize()
    tokens = np.concatenate([[1], rng.integers(6, shape[5], size=n - 1)]).astype(np.int32)
    g.prefill(tokens, want_logits=False)
    want_k, want_v = (x.reshape(shape[2], shape[6], kvd) for x in caches(g, shape))
    for t in (n - 1, n // 2 + 3, 5, 0):
        g.reset()
        bad = tokens.copy()
        bad[t] = 5
        logits, _ = g.prefill(bad)
        assert np.isnan(logits).all(), t
        for got, want in zip(caches(g, shape), (want_k, want_v)):
            got = got.reshape(shape[2], shape[6], kvd)
            np.testing.assert_array_equal(got[:, :t].view(np.uint32), want[:, :t].view(np.uint32), err_msg=str(t))
            assert np.isnan(got[1, t:n]).all(), t
    g.close()


def digit_pairs(x):
    """fp32 activations (vectors, groups, 256) as the products have them: 256 * first + second digit, 256 * third + fourth, 2^-s."""
    s = 30 - np.frexp(np.abs(x).max(axis=2, keepdims=True))[1]
    q = np.rint(np.ldexp(x.astype(np.float64), s)).astype(np.int64)
    d = (((q + 0x80808080) & 0xffffffff) ^ 0x80808080).astype(np.uint32)
    d = [(d >> np.uint32(24 - 8 * i)).astype(np.uint8).view(np.int8).astype(np.float64) for i in range(4)]
    return 256 * d[0] + d[1], 256 * d[2] + d[3], np.ldexp(np.float32(1.0), -s[:, :, 0])


@pytest.mark.parametrize("dim,heads,n", [(512, 4, 16), (512, 4, 17), (512, 4, 32), (4096, 32, 32), (4096, 32, 40), (4096, 32, 64), (4096, 32, 600), (8192, 64, 1000)])
def test_the_sums_of_a_product_are_formed_in_one_order(dim, heads, n):
    """Wv on inputs, codes and scales whose products are all exact, so that the value rows show the order of the additions to the bit.  Up
    to 32 vectors the halves of the groups are converted and added one after the other, above that the high and the low digits of a group go
    into the running sum one after the other; then the slices of K in their order."""
    vocab, kvd, ng = 512, dim // heads * 2, dim // 256
    rng = np.random.default_rng(dim + n)
    emb = np.ldexp(rng.integers(-8, 9, (vocab, dim)).astype(np.float32), rng.integers(-38, -30, (vocab, 1)))   # (nothing beside the norm's 1e-5)
    norm = rng.choice([-1.0, 127 / 128], (ng, 256)).astype(np.float32)   # (the least and the greatest code are exact)
    w = rng.integers(-128, 128, (kvd, ng, 256))
    w[..., :2] = -128, 127                                               # (a group's scale is 2^-7, its offset 0)
    g = l2j.Transformer(l2j.Config(dim, 256, 1, heads, 2, vocab, 1008, 0))
    g.fill_synthetic(9, 0.02)
    g.upload_f32(TENSOR.TOK_EMB, emb)
    g.upload_f32_quantize(TENSOR.RMS_ATT, norm)
    g.upload_f32_quantize(TENSOR.WV, np.ldexp(w, -7))
    g.finalize()
    tokens = rng.integers(2, vocab, size=n).astype(np.int32)
    g.prefill(tokens, want_logits=False)
    got = g.read(BUFFER.VCACHE, 0).reshape(-1, kvd)[:n]
    g.close()
    x = norm.reshape(-1) * (np.float32(1.0) / np.sqrt(np.float32(1e-5)) * emb[tokens])
    high, low, scale = digit_pairs(x.reshape(n, ng, 256))
    scale = np.ldexp(scale, -7)
    part = lambda d, group, k: (d[:, group, k] @ w[:, group, k].T.astype(np.float64)).astype(np.float32)   # (whole numbers: exact up to here)

    def slice_sum(g0, g1):
        f = np.zeros((n, kvd), dtype=np.float32)
        for group in range(g0, g1):
            sx = scale[:, group, None]
            for k in (slice(0, 128), slice(128, 256)) if n <= 32 else (slice(0, 256),):
                h, l = part(high, group, k), part(low, group, k)
                if n <= 32:
                    f += (h.astype(np.float64) * 65536 + l).astype(np.float32) * sx
                else:
                    f += h * (65536 * sx)
                    f += l * sx
        return f

    def want(per_slice):
        t = np.zeros((n, kvd), dtype=np.float32)
        for g0 in range(0, ng, per_slice):
            t += slice_sum(g0, min(ng, g0 + per_slice))
        return t

    if n <= 32:                                                          # (slices of four groups)
        np.testing.assert_array_equal(got.view(np.uint32), want(4).view(np.uint32))
    else:                                                                # (as many groups as the estimate for this shape picks)
        assert any(np.array_equal(got.view(np.uint32), want(per).view(np.uint32)) for per in range(1, ng + 1))


@pytest.mark.parametrize("n", [40, 64, 600])
def test_value_rows_of_small_scales_keep_their_precision(n):
    """A vector's 2^-s times a row's scale below 2^-126, in tiles of 16, 32 and 64 vectors (as for one product in test_gpu_batch.py)."""
    dim, kvd, vocab = 4096, 256, 512
    rng = np.random.default_rng(n)
    g = l2j.Transformer(l2j.Config(dim, 256, 1, 32, 2, vocab, 608, 0))
    g.fill_synthetic(9, 0.02)
    emb = np.ldexp(rng.standard_normal((vocab, dim)), -40).astype(np.float32)                 # (nothing beside the norm's 1e-5)
    g.upload_f32(TENSOR.TOK_EMB, emb)
    g.upload_f32_quantize(TENSOR.RMS_ATT, np.full(dim, 0.5))
    g.upload_f32_quantize(TENSOR.WV, np.ldexp(0.02 * rng.standard_normal((kvd, dim)), -62))
    g.finalize()
    tokens = rng.integers(2, vocab, size=n).astype(np.int32)
    g.prefill(tokens, want_logits=False)
    got = g.read(BUFFER.VCACHE, 0).reshape(-1, kvd)[:n]
    x = np.float32(0.5) * (np.float32(1.0) / np.sqrt(np.float32(1e-5)) * emb[tokens])
    want = x.astype(np.float64) @ dequantized(g, TENSOR.WV, 0, kvd, dim).T
    g.close()
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() < 3e-7, float(err.max())


def test_a_prompt_goes_through_in_smaller_passes_where_the_memory_for_a_large_one_is_missing():
    """1100 positions with room for passes of 275 instead of 550, the decode loop with option prefill likewise; other calls go on
    as before, and so does the prompt once there is room."""
    shape = (256, 28672, 1, 1, 1, 512, 1104, 1)       # (a pass of 550 rows takes 570 MB, of 275 rows 290)
    rng = np.random.default_rng(6)
    g = model(shape)
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=1099)]).astype(np.int32)
    want, _ = g.prefill(tokens)
    want_k, _ = caches(g, shape)
    single, _ = g.decode_greedy(tokens[1:], 1104)
    g.release_batch()
    g.prefill(tokens[:8])                              # the copy of the matrices and the buffers of eight rows (205 MB)
    with FullDevice(200 << 20):
        g.reset()
        got, _ = g.prefill(tokens)
        got_k, _ = caches(g, shape)
        assert rel_err(got, want.astype(np.float64)) < CLOSE and rel_err(got_k, want_k.astype(np.float64)) < CLOSE
        g.set_option("prefill", 1)
        np.testing.assert_array_equal(g.decode_greedy(tokens[1:], 1104)[0], single)
    again, _ = g.prefill(tokens)
    np.testing.assert_array_equal(again.view(np.uint32), want.view(np.uint32))
    g.close()


@pytest.mark.parametrize("n_prompt,steps", [(7, 20), (8, 9), (8, 20), (9, 20), (31, 40), (40, 37), (40, 40), (40, 41)])
def test_option_prefill_at_its_edges(orc, n_prompt, steps):
    """Prompts on both sides of the eight ids from which the option takes them at once, of no whole number of tiles, and runs that end
    inside the prompt, with it, and one step behind it: the tokens of the loop without the option."""
    shape = SHAPES[0]
    prompt = orc.synth_prompt(7, n_prompt, shape[5])
    g = model(shape)
    want, _ = g.decode_greedy(prompt, steps)
    g.reset()
    want_s, _ = g.decode_sample(prompt, steps, 0.9, 0.9, 3)
    g.set_option("prefill", 1)
    g.reset()
    np.testing.assert_array_equal(g.decode_greedy(prompt, steps)[0], want)
    g.reset()
    np.testing.assert_array_equal(g.decode_sample(prompt, steps, 0.9, 0.9, 3)[0], want_s)
    g.close()


@pytest.mark.parametrize("shape", [
    (4096, 11008, 2, 32, 32, 512, 1104, 0),     # head 128, the widths of Llama-2-7B
    (4096, 1024, 2, 64, 8, 512, 1104, 0),       # head 64, eight heads to a kv head
    (4096, 1024, 2, 16, 4, 512, 1104, 0),       # head 256
    (8192, 28672, 2, 64, 8, 512, 600, 0),       # the widths of Llama-2-70B
])
def test_wide_passes_where_their_kernels_change(shape):
    """On 256 compute units the attention of these widths has two blocks per workgroup from 257 positions on (an odd number of blocks:
    one workgroup has one), blocks of 32 positions from 545 on (head sizes 64 and 128; from 257 at 8192 wide), and the products
    change between 256 x 32 and 512 x 64 with up to sixteen columns of vectors, the last of them ragged.  Against
    position-by-position forwards: cache rows and the last position's logits; from position 0, and behind cached rows."""
    seq_len, kvd = shape[6], shape[0] // shape[3] * shape[4]
    rng = np.random.default_rng(shape[1] + shape[3])
    g = model(shape)
    tokens = np.concatenate([[1], rng.integers(2, shape[5], size=seq_len - 1)]).astype(np.int32)
    sizes = [n for n in (33, 65, 257, 272, 273, 289, 512, 513, 544, 545, 577, 600, 700, 1000, 1024, 1025) if n <= seq_len]
    want = {}
    for i, t in enumerate(tokens):
        lg = g.forward(int(t), i, want_logits=i + 1 in sizes)
        if i + 1 in sizes:
            want[i + 1] = lg
    want_kv = [x.reshape(shape[2], seq_len, kvd) for x in caches(g, shape)]
    for n in sizes:
        for first in (0, 7) if n in (273, 577, 1025) else (0,):
            g.reset()
            if first:
                g.prefill(tokens[:first], want_logits=False)
            got, _ = g.prefill(tokens[first:n], pos0=first)
            assert rel_err(got, want[n].astype(np.float64)) < CLOSE, (n, first)
            for x, y in zip(caches(g, shape), want_kv):
                x = x.reshape(shape[2], seq_len, kvd)
                assert np.abs(x[:, :n] - y[:, :n]).max() < CLOSE * np.abs(y[:, :n]).max(), (n, first)
                assert not x[:, n:].any(), (n, first)
    g.close()
