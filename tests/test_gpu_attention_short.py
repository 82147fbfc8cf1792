"""The fused schedule's attention where a head's positions are one request (up to 1024 of them for heads of 64, 512 for 128, 256 for 256): at the
edges of a request and of a lane's rows, against the reference schedule's form with the scores in LDS and on rows that must not count."""
import ctypes as C

import numpy as np
import pytest

import llama_cu_awq_amd as A
import tests.test_gpu_model as model
from llama_cu_awq_amd import synth
from llama_cu_awq_amd._lib import lib
from tests.helpers import f16, rel_l2

pytestmark = pytest.mark.gpu

takes_short = lib["_Z25awq_attention_takes_shortii"]
takes_short.argtypes, takes_short.restype = [C.c_int] * 2, C.c_bool

_short = lib["_Z26awq_launch_attention_shortP7awq_ctxPtPKtS3_S3_S1_iiiiPKi"]
_short.argtypes = [C.c_void_p] * 6 + [C.c_int] * 4 + [C.c_void_p]
_ranges = lib["_Z27awq_launch_attention_rangesP7awq_ctxPfP15HIP_vector_typeIfLj2EEPiPKtS7_S7_PtiiiiPKi"]
_ranges.argtypes = [C.c_void_p] * 3 + [C.POINTER(C.c_int)] + [C.c_void_p] * 4 + [C.c_int] * 4 + [C.c_void_p]

# heads, head size, key heads: one key head, fewer than 8, a number that is no multiple of 8
HEADS = [(4, 64, 2), (32, 64, 4), (16, 128, 1), (24, 128, 12), (8, 128, 8), (4, 256, 2), (16, 256, 16)]
POSITIONS = (0, 1, 15, 63, 64, 127, 128, 129, 255, 256, 300, 510, 511, 512, 1022, 1023)


def _transformer(ctx, heads, head, kv, seed):
    cfg = dict(dim=heads * head, hidden_dim=256, n_layers=1, n_heads=heads, n_kv_heads=kv, vocab_size=512, seq_len=1024, rope_theta=10000.0)
    return cfg, A.Transformer(ctx, image=synth.make_model_image(cfg, seed=seed))


@pytest.mark.parametrize("heads,head,kv", HEADS)
def test_against_the_reference_schedule(ctx, heads, head, kv):
    """Both round scores to fp16, and up to 256 positions the probabilities.  Activations of fp16 behind it differ by single roundings (under 1e-3
    in the norm); values that grow with the position make a row that is missed or weighted wrongly a difference of several per cent."""
    cfg, t = _transformer(ctx, heads, head, kv, 7)
    seq = cfg["seq_len"]
    rng = np.random.default_rng(heads * head + kv)
    t.buffer("key_cache", seq * kv * head * 2).write(rng.standard_normal((seq, kv * head)).astype(np.float16))
    rows = rng.standard_normal((seq, kv * head)) + 8 * np.arange(seq)[:, None] / seq - 2
    t.buffer("value_cache", seq * kv * head * 2).write(rows.astype(np.float16))
    assert [takes_short(head, n) for n in (256, 257, 512, 513, 1024, 1025)] == [True, head < 256, head < 256, head == 64, head == 64, False]
    for pos in POSITIONS:
        logits, scores = [], []
        for mode, graph in ((A.SCHEDULE_REFERENCE, False), (A.SCHEDULE_FUSED, False), (A.SCHEDULE_FUSED, True)):
            t.set_pos(pos, 7)
            t.forward_logits(use_graph=graph, mode=mode)
            ctx.sync()
            logits.append(f16(t.download("logits", cfg["vocab_size"])).astype(np.float64))
            scores.append(f16(t.download("att", heads * (pos + 1))).astype(np.float64))
        assert np.isfinite(logits[0]).all()
        for got, att in zip(logits[1:], scores[1:]):
            assert rel_l2(got, logits[0]) <= 4e-3, pos
            assert rel_l2(att, scores[0]) <= 2e-3, pos
    t.close()


@pytest.mark.parametrize("heads,head,kv", [(4, 64, 2), (16, 128, 4), (4, 256, 2)])
@pytest.mark.parametrize("pos", [0, 5, 70, 200, 260, 520])
def test_rows_past_the_position_do_not_enter(ctx, heads, head, kv, pos):
    """The first rows are read before the position is known: NaN and infinities behind it change no bit.  Those of rows that count reach
    the logits."""
    cfg, t = _transformer(ctx, heads, head, kv, 8)
    seq, row = cfg["seq_len"], kv * head
    rng = np.random.default_rng(pos)
    rows = {name: rng.standard_normal((seq, row)).astype(np.float16) for name in ("key_cache", "value_cache")}

    def logits(graph, at=None, value=0.0, names=tuple(rows)):
        for name, r in rows.items():
            r = r.copy()
            if at is not None and name in names:
                r[at] = value
            t.buffer(name, seq * row * 2).write(r)
        t.set_pos(pos, 7)
        t.forward_logits(use_graph=graph, mode=A.SCHEDULE_FUSED)
        ctx.sync()
        return f16(t.download("logits", cfg["vocab_size"])).copy()

    for graph in (False, True):
        want = logits(graph)
        assert np.isfinite(want).all()
        for value in (np.nan, np.inf):
            assert np.array_equal(logits(graph, slice(pos + 1, None), value).view(np.uint16), want.view(np.uint16))
        if pos:
            assert not np.isfinite(logits(graph, (pos - 1, row - 1), np.nan, ("key_cache",))).any()
            assert not np.isfinite(logits(graph, (0, row - 1), np.inf, ("value_cache",))).any()
    t.close()


@pytest.mark.parametrize("heads,head,kv", [(8, 64, 2)])  # (1/sqrt(head size) is exact: scores stay multiples of an eighth)
@pytest.mark.parametrize("size", [300, 512])
def test_scores_far_below_zero(ctx, heads, head, kv, size):
    """As at longer contexts: a constant added to every score changes no softmax, also where its exponentials are zero in fp32."""
    model.test_decode_scores_far_below_zero(ctx, heads, head, kv, size)


def _inputs(ctx, heads, head, kv, size, cancelling):
    """Query, keys and values of one layer.  `cancelling`: the first 32 dimensions of a key add 2^24 to its score and the next 32 take it away
    again, so that fp32 sums in another order give scores that are whole steps apart."""
    rng = np.random.default_rng(heads * head + kv + size)
    q = rng.standard_normal((heads, head)).astype(np.float16)
    k, v = (rng.standard_normal((size, kv, head)).astype(np.float16) for _ in range(2))
    if cancelling:
        q[:, [0, 32]] = 4096
        k[:, :, 0], k[:, :, 32] = 4096, -4096
    return q, k, v


@pytest.mark.parametrize("cancelling", [False, True], ids=["random", "cancelling"])
@pytest.mark.parametrize("heads,head,kv", [(32, 64, 4), (32, 128, 32), (24, 128, 12), (16, 256, 16)])
@pytest.mark.parametrize("size", [1, 64, 65, 128, 200, 256])
def test_bits_of_the_form_with_scores_in_lds(ctx, heads, head, kv, size, cancelling):
    """Up to 256 positions a sampled run takes the tokens that it takes through awq_attention: the same scores, weights and sums, bit for bit."""
    dq, dk, dv = (ctx.upload(a) for a in _inputs(ctx, heads, head, kv, size, cancelling))
    pos, got = ctx.upload(np.array([size - 1], np.int32)), []
    for short in (False, True):
        out, att = ctx.zeros(heads * head * 2), ctx.zeros(heads * size * 2)
        if short:
            assert _short(ctx.h, out.ptr, dq.ptr, dk.ptr, dv.ptr, att.ptr, heads, head, heads // kv, size, pos.ptr) == 0
        else:
            A.MultiHeadAttention(ctx, out, dq, dk, dv, att, heads, head, heads // kv, size, pos)
        got.append([d.download(np.uint16) for d in (out, att)])
    for a, b in zip(*got):
        assert np.isfinite(f16(a)).all() and np.array_equal(a, b)


@pytest.mark.parametrize("heads,head,kv,size", [(8, 64, 2, 200), (8, 64, 2, 700), (16, 128, 4, 100), (16, 128, 4, 256), (16, 128, 4, 300), (16, 128, 4, 512),
                                                (8, 256, 2, 256)])
@pytest.mark.parametrize("ranges", [False, True], ids=["short", "ranges"])
def test_every_dimension_gives_a_position_one_weight(ctx, heads, head, kv, size, ranges):
    """The lanes that share a position share its score: value rows with one number in every dimension come out with the same bits in every
    dimension."""
    q, k, v = _inputs(ctx, heads, head, kv, size, True)
    v[:] = v[:, :1, :1]
    dq, dk, dv, pos, att = (ctx.upload(a) for a in (q, k, v, np.array([size - 1], np.int32), np.zeros(heads * size, np.uint16)))
    out, stat, n = ctx.zeros(4 * heads * head * 4), ctx.zeros(4 * heads * 8), C.c_int(1)
    if ranges:
        assert _ranges(ctx.h, out.ptr, stat.ptr, C.byref(n), dq.ptr, dk.ptr, dv.ptr, att.ptr, heads, head, heads // kv, size, pos.ptr) == 0 and n.value > 1
    else:
        assert _short(ctx.h, out.ptr, dq.ptr, dk.ptr, dv.ptr, att.ptr, heads, head, heads // kv, size, pos.ptr) == 0
    got = out.download(np.uint32 if ranges else np.uint16, n.value * heads * head).reshape(-1, head)
    assert got.any() and np.array_equal(got, np.repeat(got[:, :1], head, axis=1))


@pytest.mark.parametrize("heads,head,kv,size", [(8, 64, 2, 300), (8, 64, 2, 1000), (16, 128, 4, 257), (16, 128, 4, 300), (16, 128, 4, 512)])
@pytest.mark.parametrize("ranges", [False, True], ids=["short", "ranges"])
@pytest.mark.parametrize("offset", [0, -20, -95, -150])
def test_weights_of_scores_far_below_zero(ctx, heads, head, kv, size, ranges, offset):
    """The softmax of the fp16 scores that the kernel leaves in att, over its own values, in 64 bits: also where every score's exponential
    is small, denormal or zero in fp32, and where a size's request or range ends in the middle of a wave's rows."""
    _softmax_of_published_scores(ctx, heads, head, kv, size, ranges, offset)


@pytest.mark.parametrize("heads,head,kv,size", [(8, 64, 2, 1025), (8, 64, 2, 1535), (8, 64, 2, 2100), (16, 128, 4, 700), (16, 128, 4, 1025), (16, 128, 4, 2049),
                                                (8, 256, 2, 257), (8, 256, 2, 700)])
@pytest.mark.parametrize("offset", [0, -20, -95, -150])
def test_weights_of_scores_far_below_zero_past_one_request(ctx, heads, head, kv, size, offset):
    _softmax_of_published_scores(ctx, heads, head, kv, size, True, offset)


def _softmax_of_published_scores(ctx, heads, head, kv, size, ranges, offset):
    rng = np.random.default_rng(heads * head + size)
    q = np.zeros((heads, head), np.float16)
    k = np.zeros((size, kv, head), np.float16)
    q[:, 3], k[:, :, 3] = head**0.5, rng.uniform(-4, 4, (size, kv)) + offset
    v = (rng.standard_normal((size, kv, head)) + 1).astype(np.float16)
    dq, dk, dv, pos, att = (ctx.upload(a) for a in (q, k, v, np.array([size - 1], np.int32), np.zeros(heads * size, np.uint16)))
    n = C.c_int(1)
    if ranges:
        part, stat = ctx.zeros(4 * heads * head * 4), ctx.zeros(4 * heads * 8)
        assert _ranges(ctx.h, part.ptr, stat.ptr, C.byref(n), dq.ptr, dk.ptr, dv.ptr, att.ptr, heads, head, heads // kv, size, pos.ptr) == 0 and n.value > 1
        tops, sums = np.moveaxis(stat.download(np.float32).reshape(heads, 4, 2)[:, : n.value].astype(np.float64), 2, 0)
        weight = np.exp(tops - tops.max(axis=1, keepdims=True))
        got = part.download(np.float32, n.value * heads * head).reshape(n.value, heads, head).astype(np.float64)
        got = np.einsum("hc,chd->hd", weight, got) / (weight * sums).sum(axis=1)[:, None]
    else:
        out = ctx.zeros(heads * head * 2)
        assert _short(ctx.h, out.ptr, dq.ptr, dk.ptr, dv.ptr, att.ptr, heads, head, heads // kv, size, pos.ptr) == 0
        got = f16(out.download(np.uint16)).reshape(heads, head).astype(np.float64)
    scores = f16(att.download(np.uint16)).reshape(heads, size).astype(np.float64)
    assert np.abs(scores - np.repeat(k[:, :, 3].astype(np.float64).T, heads // kv, axis=0)).max() <= 2e-3 * (4 - offset)  # (q and score rounded to fp16)
    p = np.exp(scores - scores.max(axis=1, keepdims=True))
    want = np.einsum("kgp,pkd->kgd", p.reshape(kv, -1, size) / p.sum(axis=1).reshape(kv, -1, 1), v.astype(np.float64)).reshape(heads, head)
    # weights, sums and P.V in fp32, exponentials to 2 units in the last place: 1e-6; the short form rounds its output to fp16, 2.9e-4 at most
    assert rel_l2(got, want) <= (5e-6 if ranges else 3e-4)
