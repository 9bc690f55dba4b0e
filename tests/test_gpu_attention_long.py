"""The parallel-order attention past one workgroup's prefixes: a decode step
spread over the chip or a workgroup a token's heads (prefixes beyond 768, tokens
of several conversations) and a prompt on the matrix cores in three sweeps
(prefixes beyond 1024), against the oracle's restatement of the order."""
import math

import numpy as np
import pytest

from golem_amd import capi, synth

pytestmark = pytest.mark.gpu

NAN = np.array([0x7E00], np.uint16).view(np.float16)[0]


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def _caches(g, nslots, n, kv, hd, context, exact):
    """Keys and values of n positions a conversation; the rest NaN bits."""
    k = (g.integers(-2, 3, (nslots, n, kv, hd)) * 0.25 if exact else g.standard_normal((nslots, n, kv, hd)))
    k = k.astype(np.float16)
    v = (g.standard_normal((nslots, n, kv, hd)) * 2).astype(np.float16)
    kt = np.full((nslots, kv, hd // 8, context, 8), NAN, np.float16)
    kt[:, :, :, :n] = k.reshape(nslots, n, kv, hd // 8, 8).transpose(0, 2, 3, 1, 4)
    vt = np.full((nslots, kv, hd, context), NAN, np.float16)
    vt[:, :, :, :n] = v.transpose(0, 2, 3, 1)
    return k, v, kt, vt


def _run(dev, name, qf, pos, kt, vt, heads, kv, hd, max_pos, context, slots=None, nslots=0, least=False):
    M = len(pos)
    ins = [dev.put(a) for a in (qf.view(np.int16), pos, kt.view(np.int16), vt.view(np.int16))]
    sl = None if slots is None else dev.put(slots)
    q8 = dev.full((M, heads * hd), 99, np.int8)
    sc = dev.full((M, heads * hd // 32), float("nan"))
    qs = dev.full((M, heads * hd // 32), 7777, np.int32)
    S = (max_pos + 64) // 64 * 64
    up = lambda b: (b + 255) // 256 * 256  # noqa: E731
    nw = up(M * heads * S * 4) + up(M * heads * S * 2) if least else capi.size_out(
        "gx_qwen_attention_workspace_bytes", M, heads, max_pos)
    ws = dev.empty((nw,), np.uint8)
    capi.call(name, dev.ctx.ptr, capi.vp(ins[0]), M, heads, kv, hd, max_pos, capi.vp(ins[1]), capi.vp(ins[2]),
              capi.vp(ins[3]), context, capi.vp(q8), capi.vp(sc), capi.vp(qs), capi.vp(ws), nw, capi.vp(sl), nslots)
    return dev.get(q8), dev.get(sc), dev.get(qs)


def _oracle(orc, fn, qf, k, v, pos, slots, rows, heads, kv, hd):
    lib = orc.load()
    scale = np.float32(1 / math.sqrt(float(hd)))
    want = np.zeros((len(rows), heads * hd), np.float32)
    for i, t in enumerate(rows):
        n, s = int(pos[t]) + 1, 0 if slots is None else slots[t]
        if n <= 0:
            continue
        K, V = (np.ascontiguousarray(a[s][:n].astype(np.float32)) for a in (k, v))
        scores = np.zeros(n, np.float32)
        for h in range(heads):
            query = np.ascontiguousarray(qf[t, h * hd:(h + 1) * hd].astype(np.float32))
            dst = np.zeros(hd, np.float32)
            getattr(lib, fn)(orc._p(query), orc._p(K), orc._p(V), kv, hd, h // (heads // kv), n, scale,
                             orc._p(scores), orc._p(dst))
            want[i, h * hd:(h + 1) * hd] = dst
    return want


# head width, heads, key-value heads, positions (block, run and piece edges;
# past 16,384 positions a second 256 blocks' sums, several pieces a workgroup)
DECODE = [(128, 8, 2, [768]), (128, 4, 4, [1500, 63, 64]), (64, 4, 2, [2100, 0]), (32, 8, 1, [1023, 1024, 31, 32]),
          (96, 4, 2, [801]), (32, 2, 1, [16383, 16384, 16500]), (32, 32, 8, [33000, 70, 16400, 20000])]


@pytest.mark.parametrize("hd,heads,kv,positions", DECODE)
def test_long_decode_is_the_parallel_order(dev, orc, hd, heads, kv, positions):
    """Bit for bit the restated order, whatever the launch's extent."""
    g = synth.rng(hd + len(positions))
    pos = np.array(positions, np.int32)
    n = int(pos.max()) + 1
    context = (n + 7) // 8 * 8 + 16
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, False)
    qf = (g.standard_normal((len(pos), heads * hd)) * 1.5).astype(np.float16)
    want = orc.Batch(_oracle(orc, "orc_attend_parallel", qf, k, v, pos, None, range(len(pos)), heads, kv, hd)).quantize()
    for max_pos in (n - 1, context - 1):
        q8, sc, qs = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, heads, kv, hd, max_pos, context)
        np.testing.assert_array_equal(q8, want.q_rows())
        np.testing.assert_array_equal(_bits(sc), _bits(want.scales_rows()))
        np.testing.assert_array_equal(qs, want.qsum_rows())


def test_long_decode_of_many_conversations(dev, orc):
    """Eighteen tokens of three conversations (more than the split form takes),
    two slots out of range (read inside the caches), a negative position
    (nothing visible: zeros); with the serial passes' workspace alone the call
    runs them."""
    hd, heads, kv, nslots, n, context = 64, 4, 2, 3, 800, 808
    g = synth.rng(5)
    k, v, kt, vt = _caches(g, nslots, n, kv, hd, context, False)
    pos = np.array([799, 0, -1, 64, 700, 31, 32, 767, 768, 5, 63, 127, 128, 400, 798, 255, 256, 511], np.int32)
    slots = np.array([i % 3 for i in range(18)], np.int32)
    slots[4], slots[10] = nslots + 2, -1
    qf = (g.standard_normal((18, heads * hd)) * 1.5).astype(np.float16)
    read = np.clip(slots, 0, nslots - 1)
    q8, sc, qs = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, heads, kv, hd, n - 1, context, slots, nslots)
    want = orc.Batch(_oracle(orc, "orc_attend_parallel", qf, k, v, pos, read, range(18), heads, kv, hd)).quantize()
    np.testing.assert_array_equal(q8, want.q_rows())
    np.testing.assert_array_equal(_bits(sc), _bits(want.scales_rows()))
    np.testing.assert_array_equal(qs, want.qsum_rows())
    serial = _run(dev, "gx_qwen_attention", qf, pos, kt, vt, heads, kv, hd, n - 1, context, slots, nslots)
    least = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, heads, kv, hd, n - 1, context, slots, nslots, True)
    for a, b in zip(serial, least):
        np.testing.assert_array_equal(a, b)
    assert (q8[2] == 0).all() and (sc[2] == 0).all() and (serial[0][2] == 0).all()


@pytest.mark.parametrize("M,n", [(2, 900), (4, 1024), (2, 1100)])
def test_negative_positions_of_a_lone_conversation(dev, orc, M, n):
    """To 1,024 positions a negative position sees the first one (as a prompt's
    does), past them none: zeros."""
    hd, heads, kv = 64, 4, 2
    context = (n + 7) // 8 * 8
    g = synth.rng(M + n)
    pos = np.array([n - 1, -1, -3, 0][:M], np.int32)
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, False)
    qf = g.standard_normal((M, heads * hd)).astype(np.float16)
    q8, sc, qs = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, heads, kv, hd, n - 1, context)
    seen = np.maximum(pos, 0) if n <= 1024 else pos
    want = orc.Batch(_oracle(orc, "orc_attend_parallel", qf, k, v, seen, None, range(M), heads, kv, hd)).quantize()
    np.testing.assert_array_equal(q8, want.q_rows())
    np.testing.assert_array_equal(_bits(sc), _bits(want.scales_rows()))
    np.testing.assert_array_equal(qs, want.qsum_rows())


def test_rows_alone_of_a_lone_conversation(dev):
    """With the serial passes' workspace alone, two tokens to 1,024 positions
    run as the end of a prompt."""
    hd, heads, kv, n, context = 64, 4, 2, 900, 904
    g = synth.rng(17)
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, False)
    qf = g.standard_normal((6, heads * hd)).astype(np.float16)
    pos = np.arange(n - 6, n, dtype=np.int32)
    args = (kt, vt, heads, kv, hd, n - 1, context)
    prompt = _run(dev, "gx_qwen_attention_parallel", qf, pos, *args)
    two = _run(dev, "gx_qwen_attention_parallel", np.ascontiguousarray(qf[4:]), pos[4:].copy(), *args, least=True)
    for a, b in zip(prompt, two):
        np.testing.assert_array_equal(a[4:].view(np.uint8), b.view(np.uint8))


# head width, heads, key-value heads, tokens, longest prefix.  A workgroup a
# token's heads: one, two and four heads each, their scores in LDS and (past
# 2,016 positions of four heads, 4,032 of two, 8,064 of one) in the caller's
# rows; a head's elements 32 a workgroup.  The positions over the chip: a
# workgroup a piece, and several pieces a workgroup
FORMS = [(128, 8, 1, 20, 900), (64, 16, 4, 20, 800), (32, 16, 8, 20, 4100), (128, 32, 8, 28, 800),
         (96, 32, 8, 26, 2310), (64, 2, 1, 17, 8200), (96, 4, 4, 3, 1000), (64, 32, 8, 16, 1024), (128, 32, 8, 8, 1000),
         (64, 8, 1, 16, 1100), (32, 32, 32, 16, 2400)]


@pytest.mark.parametrize("hd,heads,kv,M,n", FORMS)
def test_long_decode_forms(dev, orc, hd, heads, kv, M, n):
    """Bit for bit the restated order in either form, over prefixes of no
    position, one, the edges of runs, blocks and chunks, all; slots out of
    range read inside the caches."""
    g = synth.rng(hd + M + n)
    nslots, context = 2, (n + 7) // 8 * 8
    edges = [n - 1, -1, 0, 31, 32, 63, 64, 127, 128, 159, 160, 255, 256, 511, 512, 575, 576, n // 2, n - 33, n - 64]
    pos = np.array([edges[i] if i < len(edges) else int(g.integers(0, n)) for i in range(M)], np.int32)
    slots = np.array([nslots + 5 if i == 3 else -2 if i == 2 else i % nslots for i in range(M)], np.int32)
    k, v, kt, vt = _caches(g, nslots, n, kv, hd, context, False)
    qf = (g.standard_normal((M, heads * hd)) * 1.5).astype(np.float16)
    read = np.clip(slots, 0, nslots - 1)
    q8, sc, qs = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, heads, kv, hd, n - 1, context, slots, nslots)
    want = orc.Batch(_oracle(orc, "orc_attend_parallel", qf, k, v, pos, read, range(M), heads, kv, hd)).quantize()
    np.testing.assert_array_equal(q8, want.q_rows())
    np.testing.assert_array_equal(_bits(sc), _bits(want.scales_rows()))
    np.testing.assert_array_equal(qs, want.qsum_rows())


# head width, heads, key-value heads, M, first position, context: few tiles
# (eight wavefronts) and many (four), ragged tiles, one token past 1024; block
# sums past 64 KB of LDS, and the most that fit it
PROMPT = [(128, 4, 1, 33, 1100, 1144), (64, 4, 2, 70, 990, 1064), (32, 8, 1, 5, 1020, 1032), (96, 4, 4, 64, 1500, 1568),
          (32, 32, 8, 544, 600, 1160), (128, 32, 8, 530, 500, 1032), (32, 2, 1, 5, 33000, 33008),
          (64, 2, 2, 6, 76794, 76800)]


@pytest.mark.parametrize("hd,heads,kv,M,start,context", PROMPT)
def test_long_prompt_on_exact_scores(dev, orc, hd, heads, kv, M, start, context):
    """Queries and keys on a grid of 1/4, so that scores and probabilities are
    the restated order's bits: only the value sums' order differs, 1e-5 of RMS
    at most (1,600 products of fp32 sums; about 1e-6 expected), which moves a
    Q8_0 value (a step is about 1/40 of RMS) in at most one of 1,000 and a
    scale (fp16) by at most a step."""
    g = synth.rng(M + hd + start)
    n = start + M
    pos = np.arange(start, n, dtype=np.int32)
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, True)
    qf = (g.integers(-2, 3, (M, heads * hd)) * 0.25).astype(np.float16)
    q8, sc, qs = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, heads, kv, hd, n - 1, context)
    rows = [t for t in sorted({0, 1, 15, 31, 32, M // 2, M - 2, M - 1}) if t < M]
    heads_w = _oracle(orc, "orc_attend_parallel", qf, k, v, pos, None, rows, heads, kv, hd)
    want = orc.Batch(heads_w).quantize()
    dq = q8[rows].astype(np.int32) - want.q_rows().astype(np.int32)
    assert np.abs(dq).max() <= 1 and np.count_nonzero(dq) <= max(3, dq.size // 1000)
    assert np.abs(sc[rows] / want.scales_rows() - 1).max() <= 2.0 ** -10
    np.testing.assert_array_equal(qs, q8.reshape(M, -1, 32).astype(np.int32).sum(2))


def test_prompt_past_the_sweeps_runs_the_serial_passes(dev):
    """A position more than the block sums' LDS holds."""
    hd, heads, kv, M, n = 32, 2, 1, 5, 76801
    context = (n + 7) // 8 * 8
    g = synth.rng(8)
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, False)
    qf = g.standard_normal((M, heads * hd)).astype(np.float16)
    pos = np.arange(n - M, n, dtype=np.int32)
    args = (qf, pos, kt, vt, heads, kv, hd, n - 1, context)
    for a, b in zip(_run(dev, "gx_qwen_attention_parallel", *args), _run(dev, "gx_qwen_attention", *args)):
        np.testing.assert_array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("hd", [32, 128])
def test_long_prompt_does_not_depend_on_its_batch(dev, hd):
    """Past 1,024 positions a prompt's token gets the same bits whether its
    batch is the whole document (four wavefronts a workgroup) or its last
    tokens (eight, and other tiles)."""
    heads, kv, n, few = 16, 2, 1060, 41
    context = (n + 7) // 8 * 8
    g = synth.rng(hd + 7)
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, False)
    qf = g.standard_normal((n, heads * hd)).astype(np.float16)
    pos = np.arange(n, dtype=np.int32)
    args = (kt, vt, heads, kv, hd, n - 1, context)
    whole = _run(dev, "gx_qwen_attention_parallel", qf, pos, *args)
    last = _run(dev, "gx_qwen_attention_parallel", np.ascontiguousarray(qf[-few:]), pos[-few:].copy(), *args)
    for a, b in zip(whole, last):
        np.testing.assert_array_equal(a[-few:].view(np.uint8), b.view(np.uint8))


# LDS and sweeps of eight and (33 tiles of 16 heads) four wavefronts
WILD = [(128, 1100, 70), (64, 600, 70), (128, 0, 70), (64, 300, 70), (96, 505, 70), (32, 700, 70), (32, 0, 1040),
        (128, 40, 1060)]


@pytest.mark.parametrize("hd,start,M", WILD)
def test_long_prompt_keeps_later_infinities_out(dev, hd, start, M):
    """An infinite and a NaN value of two tokens in mid-tile: the tokens before
    them get the bits they get without them, the tokens after them everywhere
    but in the blocks of the two elements."""
    heads, kv = 16, 2
    n = start + M
    context = (n + 7) // 8 * 8
    g = synth.rng(hd)
    k, v, kt, vt = _caches(g, 1, n, kv, hd, context, False)
    qf = g.standard_normal((M, heads * hd)).astype(np.float16)
    pos = np.arange(start, n, dtype=np.int32)
    args = (heads, kv, hd, n - 1, context)
    clean = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, *args)
    first, second = 13, 41  # tokens, of the first and the second tile
    vt[0, 0, 5, start + first] = np.inf
    vt[0, 1, hd - 1, start + second] = NAN
    wild = _run(dev, "gx_qwen_attention_parallel", qf, pos, kt, vt, *args)
    blocks = np.arange(heads * hd // 32) * 32
    own = (blocks % hd + 31 - hd + 1 == 0), (blocks % hd == 0)  # the last block of a head, the first
    hit = np.zeros((M, blocks.size), bool)
    hit[first:] |= (blocks // hd < heads // kv) & own[1]
    hit[second:] |= (blocks // hd >= heads // kv) & own[0]
    for a, b in zip(clean, wild):
        a, b = (_bits(u).reshape(M, blocks.size, -1) if u.dtype == np.float32 else u.reshape(M, blocks.size, -1)
                for u in (a, b))
        np.testing.assert_array_equal(a[~hit], b[~hit])
    # the infinity reaches its block's scale at every later token (a Q8_0
    # block's peak passes a NaN by, so the other's says nothing)
    block = hit[M - 1] & (blocks // hd < heads // kv)
    assert np.isinf(wild[1][first:, block]).all()
