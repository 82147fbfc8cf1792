"""The batched int4 GEMM in each of its forms (one workgroup tile of 32, 64, 96 or 128 rows by 64, 128 or 256 columns, K
slices inside a workgroup and over workgroups): rows and K ranges around tile ends, K that is no multiple of a quantisation
group, K past eight groups (scales and zeros travel for eight at a time), against the product in 64 bits.

Bar: the weights are exact fp16 values, sums are fp32 and the result is rounded once: rel-L2 2.1e-4 by the rounding alone;
1e-3 as for the other GEMM tests."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import llama_cu_awq_amd as A
from llama_cu_awq_amd import synth
from llama_cu_awq_amd._lib import QWeightC, lib
from tests.helpers import f16, rel_l2

pytestmark = pytest.mark.gpu

# per form (rows, columns of a workgroup's tile): products whose K is one piece, and parts of K that meet in the workspace
SHAPES = {
    (32, 64): {1: [(31, 160, 384), (32, 1120, 1152), (64, 1184, 8192)], 2: [(33, 2048, 128)], 3: [(16, 4128, 256)], 4: [(1, 4096, 384)]},
    (64, 64): {1: [(65, 512, 6144), (97, 416, 4224), (129, 2080, 4096)], 2: [(33, 5152, 6144)], 3: [(33, 3072, 1152)], 4: [(97, 4096, 384)]},
    (64, 128): {1: [(65, 256, 6144), (65, 160, 6144), (300, 1056, 4096), (257, 1184, 12288)], 2: [(129, 8224, 9216)], 3: [(513, 4128, 2048)]},
    (64, 256): {1: [(257, 128, 12288), (300, 96, 12288), (385, 1184, 18432)], 3: [(289, 8192, 8192)]},
    (96, 256): {1: [(700, 128, 6144), (513, 96, 8192), (700, 1152, 6144)], 2: [(898, 6176, 2304)], 3: [(65, 4128, 18432)], 4: [(65, 6176, 12288)]},
    (128, 256): {1: [(385, 128, 16384), (385, 96, 16384), (513, 1120, 12288)], 3: [(324, 6176, 6144)]},
    (128, 128): {1: [(1, 128, 128), (385, 1184, 8192)], 2: [(324, 4096, 3072), (65, 4128, 12288)]},
}
CASES = [(*shape, form, parts) for form, by_parts in SHAPES.items() for parts, shapes in by_parts.items() for shape in shapes]


@pytest.mark.parametrize("M,K,N,form,parts", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_against_fp64(ctx, M, K, N, form, parts):
    rows, cols, _, split = A.gemm_form(M, K, N)
    assert ((rows, cols), split) == (form, parts)
    key = synth.stream_key(52, M, K, N)
    w, z, s = synth.make_qweight(key, K, N)
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K)
    resid = synth.normal_f16(synth.stream_key(key, "r"), M * N)
    qw, da = A.QWeight.upload(ctx, w, z, s), ctx.upload(a)
    w16 = synth.dequantize(w, z, s, K).astype(np.float32).astype(np.float16).astype(np.float64)
    truth = a.astype(np.float64).reshape(M, K) @ w16.T
    outs = []
    for fn in (A.gemm_q, A.gemm_q_static, A.gemm_q):  # the arrival counters are back at zero for the second call
        dout = ctx.zeros(M * N * 2)
        fn(ctx, dout, N, da, K, M, qw, K, N)
        outs.append(dout.download(np.uint16))
    got = f16(outs[0]).reshape(M, N)
    assert rel_l2(got, truth) <= 1e-3
    assert rel_l2(got[-1], truth[-1]) <= 1e-3 and rel_l2(got[:, -32:], truth[:, -32:]) <= 1e-3
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    dout = ctx.upload(resid)
    A.gemm_q(ctx, dout, N, da, K, M, qw, K, N, accum=True)
    assert rel_l2(f16(dout.download(np.uint16)).reshape(M, N), truth + resid.astype(np.float64).reshape(M, N)) <= 1e-3


# the row form and the 128 x 128 kernel; K that ends in the middle of a step (33 units of 32) or of a quantisation group
@pytest.mark.parametrize("M,K,N,form", [(40, 1056, 256, (32, 64)), (512, 1056, 8192, (128, 128)), (512, 1088, 8192, (128, 128)), (512, 1120, 8192, (128, 128))])
@pytest.mark.parametrize("last", [False, True], ids=["first-column", "last-column"])
def test_infinite_activation_stays_in_its_row(ctx, M, K, N, form, last):
    """K that ends in the middle of a step: nothing of a neighbouring row (or of the memory behind the last one) enters."""
    assert A.gemm_form(M, K, N)[:2] == form
    col = K - 1 if last else 0
    key = synth.stream_key(53, M, K, N)
    w, z, s = synth.make_qweight(key, K, N)
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K).copy()
    qw = A.QWeight.upload(ctx, w, z, s)
    outs = []
    for value in (None, np.float16(np.inf)):
        b = a.copy()
        if value is not None:
            b[20, col] = value
        dout = ctx.zeros(M * N * 2)
        A.gemm_q(ctx, dout, N, ctx.upload(b.reshape(-1)), K, M, qw, K, N)
        outs.append(dout.download(np.uint16).reshape(M, N))
    rest = [m for m in range(M) if m != 20]
    assert np.array_equal(outs[0][rest], outs[1][rest])
    w16 = synth.dequantize(w, z, s, K).astype(np.float32)
    got = f16(outs[1][20])
    assert np.array_equal(np.isposinf(got), w16[:, col] > 0) and np.array_equal(np.isneginf(got), w16[:, col] < 0)


@pytest.mark.parametrize("M,K,N,form", [(40, 1056, 256, (32, 64)), (65, 1120, 6144, (64, 64)), (300, 1056, 4096, (64, 128)), (300, 96, 12288, (64, 256)), (700, 1120, 6144, (96, 256)),
                                        (513, 1120, 12288, (128, 256)), (512, 1056, 8192, (128, 128))])
def test_weights_past_the_range_of_fp16(ctx, M, K, N, form):
    """(q - z) * s beyond 65504 is an infinite weight; against positive activations its column is infinite, and what a load
    past the end of a row brings in does not make it NaN."""
    assert A.gemm_form(M, K, N)[:2] == form
    key = synth.stream_key(56, M, K, N)
    w, z, s = synth.make_qweight(key, K, N)
    pwh, pzh, sh = synth.strides(K)
    w, z, s = w.reshape(N, pwh).copy(), z.reshape(N, pzh).copy(), s.reshape(N, sh).copy()
    w[5, : K // 8] = 0xFFFFFFFF
    z[5] = 0
    s[5, -1] = np.float16(6000.0)  # 15 * 6000, in the last group only
    a = np.abs(synth.normal_f16(synth.stream_key(key, "a"), M * K)) + np.float16(0.5)
    dout = ctx.zeros(M * N * 2)
    A.gemm_q(ctx, dout, N, ctx.upload(a.astype(np.float16)), K, M, A.QWeight.upload(ctx, w.reshape(-1), z.reshape(-1), s.reshape(-1)), K, N)
    got = f16(dout.download(np.uint16)).reshape(M, N)
    assert np.isposinf(got[:, 5]).all() and np.isfinite(np.delete(got, 5, 1)).all()


# 64-wide heads, sizes at which the QKV and gate/up products take the 64 to 128 row forms by 128 and 256 columns (passes of up to 128
# rows go in the few-row form; the row forms' epilogues at few rows are held against 64-bit products below)
SMALL = dict(dim=2048, hidden_dim=5632, n_layers=2, n_heads=32, n_kv_heads=4, vocab_size=512, seq_len=1280, rope_theta=10000.0)


@pytest.fixture(scope="module")
def small(ctx):
    img = synth.make_model_image(SMALL, seed=54, scale_mult=0.25)
    prompt = synth.prompt_tokens(54, 1000, SMALL["vocab_size"])
    t = A.Transformer(ctx, image=img)
    t.reset(prompt)
    for i in range(1000):
        t.forward(i == 999, use_graph=True)
    ctx.sync()
    want = _rows(t, 1000)
    t.close()
    return img, prompt, want


def _rows(t, n):
    kv_dim = SMALL["dim"] * SMALL["n_kv_heads"] // SMALL["n_heads"]
    size = SMALL["n_layers"] * SMALL["seq_len"] * kv_dim
    return [f16(t.download(name, size)).reshape(SMALL["n_layers"], SMALL["seq_len"], kv_dim)[:, :n].copy() for name in ("key_cache", "value_cache")]


@pytest.mark.parametrize("parts", [(20, 45), (100, 129), (300, 400), (1000,)], ids=str)
def test_prefill_epilogues_against_token_by_token(ctx, small, parts):
    img, prompt, want = small
    n = sum(parts)
    t = A.Transformer(ctx, image=img)
    t.reset(prompt[:n])
    for p in parts:
        t.prefill(p, gen_token=False)
    ctx.sync()
    got = _rows(t, n)
    t.close()
    for a, b in zip(got, want):
        for l in range(SMALL["n_layers"]):
            assert rel_l2(a[l], b[l][:n]) <= 1e-2, l
            assert rel_l2(a[l][-3:], b[l][n - 3 : n]) <= 1e-2, l


class _Plan(C.Structure):  # of the row forms: which, into how many parts K is split over workgroups, the time expected
    _fields_ = [("form", C.c_int), ("parts", C.c_int), ("us", C.c_float)]


_plan = lib["_Z18awq_plan_gemm_rowsiiiibb"]  # compute units, rows, K, columns / 64, may split, the parts stay apart
_plan.argtypes, _plan.restype = [C.c_int] * 4 + [C.c_bool] * 2, _Plan
_resid = lib["_Z21awq_launch_gemm_residP7awq_ctxPtPKtiiPK11awq_qweightiiPi"]
_resid.argtypes = [C.c_void_p] * 3 + [C.c_int] * 2 + [C.POINTER(QWeightC)] + [C.c_int] * 2 + [C.POINTER(C.c_int)]
_norm_parts = lib["_Z24awq_launch_rmsnorm_partsP7awq_ctxPtS1_PKtiiii"]
_norm_parts.argtypes = [C.c_void_p] * 4 + [C.c_int] * 4


# (rows, K, columns) by the parts that K is split into: every form that splits, single and ragged rows, columns that end in the
# first piece of a thread, in its second and past both (more than 8192: read and written twice)
LEFT = {2: [(1, 2048, 128), (257, 2048, 1024), (385, 3072, 4096), (129, 2048, 12288), (200, 4096, 12288)],
        3: [(1, 3072, 128), (450, 3072, 384), (97, 2048, 8320), (150, 6144, 12288), (129, 6144, 9216)],
        4: [(1, 4096, 128), (321, 4096, 384), (257, 4096, 2048), (33, 4096, 8320), (97, 4096, 12288)]}


@pytest.mark.parametrize("perm", [0, 1])
@pytest.mark.parametrize("M,K,N,parts", [(*shape, n) for n, shapes in LEFT.items() for shape in shapes])
def test_parts_left_to_the_norm(ctx, M, K, N, parts, perm):
    """A residual product whose parts the norm adds up, against the one whose parts meet in the launch (held against 64 bits
    above) and the plain norm behind it.  Both round the same fp32 sum once: apart from its order, under 1e-6, they differ where
    that crosses a rounding, one element in some thousand by 2^-11: 1e-4."""
    key = synth.stream_key(59, M, K, N)
    qw = A.QWeight.upload(ctx, *synth.make_qweight(key, K, N))
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K // 8, 8)
    da, da_perm = (ctx.upload(np.ascontiguousarray(v).reshape(-1)) for v in (a, a[:, :, [0, 4, 1, 5, 2, 6, 3, 7]]))
    x = synth.normal_f16(synth.stream_key(key, "x"), M * N)
    norm = ctx.upload(synth.normal_f16(synth.stream_key(key, "n"), N, 1.0, 0.02))
    outs = []
    for split in (False, True):
        dx, do, left = ctx.upload(x), ctx.zeros(M * N * 2), C.c_int(0)
        if split:
            assert _resid(ctx.h, dx.ptr, da_perm.ptr, K, M, C.byref(qw.c), K, N, C.byref(left)) == 0 and left.value == parts
        else:
            A.gemm_q(ctx, dx, N, da, K, M, qw, K, N, accum=True)
        assert _norm_parts(ctx.h, do.ptr, dx.ptr, norm.ptr, N, M, perm, left.value) == 0
        outs.append([f16(d.download(np.uint16)).reshape(M, N) for d in (dx, do)])
    for got, want in zip(outs[1], outs[0]):
        assert np.isfinite(want).all() and rel_l2(got, want) <= 1e-4
        assert rel_l2(got[-1], want[-1]) <= 1e-3 and rel_l2(got[:, -8:], want[:, -8:]) <= 1e-3


_qkv = lib["_Z19awq_launch_gemm_qkvP7awq_ctxPtS1_S1_PKtiiPK11awq_qweightS6_S6_iiiiPK15HIP_vector_typeIfLj2EEfibb"]
_qkv.argtypes = [C.c_void_p] * 5 + [C.c_int] * 2 + [C.POINTER(QWeightC)] * 3 + [C.c_int] * 4 + [C.c_void_p, C.c_float, C.c_int, C.c_bool, C.c_bool]
_ffn = lib["_Z19awq_launch_gemm_ffnP7awq_ctxPtPKtiiPK11awq_qweightS6_iibbb"]
_ffn.argtypes = [C.c_void_p] * 3 + [C.c_int] * 2 + [C.POINTER(QWeightC)] * 2 + [C.c_int] * 2 + [C.c_bool] * 3
_plan_few = lib["_Z17awq_plan_gemm_fewiiiib"]  # compute units, rows, K, columns, may split (its fields: see _Plan)
_plan_few.argtypes, _plan_few.restype = [C.c_int] * 4 + [C.c_bool], _Plan
_takes_few = lib["_Z21awq_prefill_takes_fewP7awq_ctxiiii"]
_takes_few.argtypes, _takes_few.restype = [C.c_void_p] + [C.c_int] * 4, C.c_bool
_tile = lib["_Z13awq_rows_formiPi"]
_tile.argtypes, _tile.restype = [C.c_int, C.POINTER(C.c_int)], None


def _form(M, K, N):
    """Tile and parts of K of a product that is not a single matrix."""
    plan, tile = _plan(256, M, K, N // 64, True, False), (C.c_int * 3)()
    _tile(plan.form, tile)
    return (tile[0], tile[1]), plan.parts


# up to 128 rows, where passes whose products do not take the few-row form (matrices of 8192 by 28672, say) run QKV and gate/up: whole K
# and parts of it that meet in the launch.  (rows, K, query columns, key and value columns, head size, tile, parts)
QKV = [(20, 256, 128, 128, 64, (32, 64), 1), (1, 2048, 128, 128, 128, (32, 64), 2), (37, 3072, 128, 128, 64, (32, 64), 3), (33, 4096, 128, 128, 128, (32, 64), 4),
       (64, 512, 6400, 1024, 256, (64, 64), 1), (65, 8192, 2048, 384, 128, (64, 64), 2), (48, 3072, 512, 256, 256, (64, 64), 3), (128, 4096, 640, 128, 64, (64, 64), 4),
       (37, 256, 6272, 1024, 128, (64, 128), 1), (100, 4096, 6272, 1024, 64, (64, 128), 3)]
# (rows, K, hidden, tile, parts)
FFN = [(20, 256, 256, (32, 64), 1), (1, 2048, 256, (32, 64), 2), (33, 3072, 256, (32, 64), 3), (37, 4096, 256, (32, 64), 4), (64, 512, 4224, (64, 64), 1),
       (65, 8192, 1408, (64, 64), 2), (48, 3072, 512, (64, 64), 3), (128, 4096, 384, (64, 64), 4), (37, 256, 4224, (64, 128), 1), (100, 4096, 4224, (64, 128), 3)]


def _matrix(ctx, key, K, N):
    """On the device, and as the kernels multiply it."""
    w, z, s = synth.make_qweight(key, K, N)
    return A.QWeight.upload(ctx, w, z, s), synth.dequantize(w, z, s, K).astype(np.float32).astype(np.float16).astype(np.float64)


def _rows_in_packed_order(ctx, key, M, K):
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K)
    return ctx.upload(np.ascontiguousarray(a.reshape(M, K // 8, 8)[:, :, [0, 4, 1, 5, 2, 6, 3, 7]]).reshape(-1)), a.astype(np.float64).reshape(M, K)


def _near(got, want):
    assert rel_l2(got, want) <= 4e-4
    for at in (np.s_[-1], np.s_[0], np.s_[:, -32:], np.s_[:, :32]):
        assert rel_l2(got[at], want[at]) <= 1e-3


@pytest.mark.parametrize("M,K,Nq,Nkv,head,tile,parts", QKV)
def test_qkv_of_few_rows_against_fp64(ctx, M, K, Nq, Nkv, head, tile, parts):
    """Rotated q and k, v as it is, cache rows from a position on.  q and k are rounded to fp16 before the rotation and behind it, v once
    (2.1e-4 in the norm each, 3.0e-4 together)."""
    assert _form(M, K, Nq + 2 * Nkv) == (tile, parts)
    key, pos0 = synth.stream_key(66, M, K, Nq), 5
    mats = [_matrix(ctx, synth.stream_key(key, name), K, n) for name, n in (("q", Nq), ("k", Nkv), ("v", Nkv))]
    da, a = _rows_in_packed_order(ctx, key, M, K)
    angle = np.random.default_rng(M + Nq).uniform(0, 2 * np.pi, (pos0 + M, head // 2))
    rope = np.stack([np.cos(angle), np.sin(angle)], axis=-1).astype(np.float32)
    dr, runs = ctx.upload(rope), []
    for _ in range(2):  # (the arrival counters are back at zero for the second launch)
        outs = [ctx.upload(np.full((first + M + 1) * n, 0xFFFF, np.uint16)) for n, first in ((Nq, 0), (Nkv, pos0), (Nkv, pos0))]
        assert _qkv(ctx.h, *(o.ptr for o in outs), da.ptr, K, M, *(C.byref(m.c) for m, _ in mats), K, Nq, Nkv, head, dr.ptr, 10000.0, pos0, True, False) == 0
        runs.append([o.download(np.uint16) for o in outs])
    for i, (n, first) in enumerate(((Nq, 0), (Nkv, pos0), (Nkv, pos0))):
        assert np.array_equal(runs[0][i], runs[1][i])
        bits = runs[0][i].reshape(-1, n)
        assert (bits[:first] == 0xFFFF).all() and (bits[first + M :] == 0xFFFF).all()
        want = a @ mats[i][1].T
        if i < 2:
            x, y = (want.reshape(M, -1, 2, head // 2)[:, :, j] for j in (0, 1))
            c, s = (rope[pos0:, None, :, j].astype(np.float64) for j in (0, 1))
            want = np.stack([x * c - y * s, x * s + y * c], axis=2).reshape(M, n)
        _near(f16(bits[first : first + M]).astype(np.float64), want)


@pytest.mark.parametrize("M,K,N,tile,parts", FFN)
def test_gate_and_up_of_few_rows_against_fp64(ctx, M, K, N, tile, parts):
    """silu(gate) * up in fp32, rounded once (2.1e-4 in the norm), every 8 columns in the order that a packed dword unpacks in."""
    assert _form(M, K, 2 * N) == (tile, parts)
    key = synth.stream_key(67, M, K, N)
    (gate, gate64), (up, up64) = (_matrix(ctx, synth.stream_key(key, name), K, N) for name in ("gate", "up"))
    (da, a), runs = _rows_in_packed_order(ctx, key, M, K), []
    for _ in range(2):
        dh = ctx.zeros(M * N * 2)
        assert _ffn(ctx.h, dh.ptr, da.ptr, K, M, C.byref(gate.c), C.byref(up.c), K, N, True, True, False) == 0
        runs.append(dh.download(np.uint16))
    assert np.array_equal(*runs)
    g, u = (a @ m.T for m in (gate64, up64))
    _near(f16(runs[0]).reshape(M, N // 8, 8)[:, :, [0, 2, 4, 6, 1, 3, 5, 7]].reshape(M, N).astype(np.float64), g / (1 + np.exp(-g)) * u)


# (looked up through the library: the HIP runtime it is linked with)
def _hip(name, *args):
    assert getattr(lib, name)(*args) == 0, name


def test_split_workspace_made_while_recording(ctx):
    """The first product of a context, recorded: the arrival counters are clear before the graph has run, and nothing but the
    product is recorded."""
    M, K, N = 33, 2048, 128
    assert A.gemm_form(M, K, N)[3] > 1
    key = synth.stream_key(57, M, K, N)
    qw = A.QWeight.upload(ctx, *synth.make_qweight(key, K, N))
    a = [ctx.upload(synth.normal_f16(synth.stream_key(key, i), M * K)) for i in range(2)]
    out = [ctx.zeros(M * N * 2) for _ in a]
    fresh = A.Context(0)
    ctx.sync()
    stream, graph, runnable, nodes = C.c_void_p(lib.awq_ctx_stream(fresh.h)), C.c_void_p(), C.c_void_p(), C.c_size_t()
    _hip("hipStreamBeginCapture", stream, 2)  # relaxed: allocations are allowed
    A.gemm_q(fresh, out[0], N, a[0], K, M, qw, K, N)
    _hip("hipStreamEndCapture", stream, C.byref(graph))
    _hip("hipGraphGetNodes", graph, None, C.byref(nodes))
    assert nodes.value == 1
    _hip("hipGraphInstantiate", C.byref(runnable), graph, None, None, C.c_size_t(0))
    want = []
    for x in a:
        d = ctx.zeros(M * N * 2)
        A.gemm_q_static(ctx, d, N, x, K, M, qw, K, N)
        want.append(d.download(np.uint16))
    for _ in range(3):  # an eager product before the first replay and between the others
        A.gemm_q(fresh, out[1], N, a[1], K, M, qw, K, N)
        fresh.sync()
        assert np.array_equal(out[1].download(np.uint16), want[1])
        _hip("hipGraphLaunch", runnable, stream)
        fresh.sync()
        assert np.array_equal(out[0].download(np.uint16), want[0])
        for d in out:
            d.write(np.zeros(M * N, np.uint16))
    _hip("hipGraphExecDestroy", runnable)
    _hip("hipGraphDestroy", graph)
    fresh.close()


@pytest.mark.parametrize("few,n,kv,hidden", [(True, 37, 4, 2048), (False, 100, 1, 1024)])
def test_short_prefill_recorded_after_a_long_one(few, n, kv, hidden):
    """1100 rows by 4096 columns split no K, the short prompt's do: 37 rows in the few-row form (O and down of the first of two layers,
    whose parts the norm adds up), 100 in the row forms (gate/up, whose parts meet in the launch, and O, whose parts the norm adds up).
    What that takes is there before the short prompt is recorded."""
    cfg = dict(dim=4096, hidden_dim=hidden, n_layers=2, n_heads=32, n_kv_heads=kv, vocab_size=512, seq_len=1280, rope_theta=10000.0)
    img = synth.make_model_image(cfg, seed=55, scale_mult=0.25)
    prompt = synth.prompt_tokens(55, 1100 + n, cfg["vocab_size"])
    ctx = A.Context(0)
    t = A.Transformer(ctx, image=img)
    kv_dim = kv * 128

    def caches():
        return [t.download(name, size) for name, size in (("key_cache", 2 * cfg["seq_len"] * kv_dim), ("value_cache", 2 * cfg["seq_len"] * kv_dim), ("logits", 512))]

    stream, graph, runnable = C.c_void_p(lib.awq_ctx_stream(ctx.h)), C.c_void_p(), C.c_void_p()
    t.reset(prompt)
    t.prefill(1100, gen_token=False)
    _hip("hipStreamBeginCapture", stream, 0)
    t.prefill(n, gen_token=False)
    _hip("hipStreamEndCapture", stream, C.byref(graph))
    _hip("hipGraphInstantiate", C.byref(runnable), graph, None, None, C.c_size_t(0))
    recorded = []
    for _ in range(3):
        _hip("hipGraphLaunch", runnable, stream)
        ctx.sync()
        recorded.append(caches())
    t.reset(prompt)
    t.prefill(1100, gen_token=False)
    t.prefill(n, gen_token=False)
    ctx.sync()
    want = caches()
    for got in recorded:
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
        for b in want[:2]:
            assert f16(b).reshape(2, -1, kv_dim)[:, 1100 : 1100 + n].any(axis=2).all()
    assert _takes_few(ctx.h, n, 4096, kv_dim, hidden) == few
    if few:
        assert all(_plan_few(256, n, K, 4096, True).parts > 1 for K in (4096, hidden))
    else:
        assert _form(n, 4096, 2 * hidden)[1] > 1 and _plan(256, n, 4096, 4096 // 64, True, True).parts > 1
    _hip("hipGraphExecDestroy", runnable)
    _hip("hipGraphDestroy", graph)
    t.close()
    ctx.close()


# hipMalloc fails for the split-K workspace's 32 MiB and its counters, and for nothing else, with the runtime's own error
NO_WORKSPACE = """
#include <dlfcn.h>
#include <stddef.h>
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so", RTLD_NOW), "hipMalloc");
    return real(p, n == ((size_t)32 << 20) + 1024 ? (size_t)1 << 60 : n);
}
"""
WITHOUT_WORKSPACE = """
import ctypes as C, sys
C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
import numpy as np
import llama_cu_awq_amd as A
from llama_cu_awq_amd import synth
from llama_cu_awq_amd._lib import QWeightC, lib
M, K, N = 900, 11008, 4096
ctx = A.Context(0)
key = synth.stream_key(58, M, K, N)
qw = A.QWeight.upload(ctx, *synth.make_qweight(key, K, N))
a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K // 8, 8)
x = synth.normal_f16(synth.stream_key(key, "x"), M * N)
rows = [ctx.upload(np.ascontiguousarray(v).reshape(-1)) for v in (a, a[:, :, [0, 4, 1, 5, 2, 6, 3, 7]])]
outs = [ctx.upload(x) for _ in rows]
A.gemm_q_static(ctx, outs[0], N, rows[0], K, M, qw, K, N, accum=True)
reserve, resid = lib["_Z26awq_reserve_gemm_workspaceP7awq_ctx"], lib["_Z21awq_launch_gemm_residP7awq_ctxPtPKtiiPK11awq_qweightiiPi"]
reserve.argtypes = [C.c_void_p]
resid.argtypes = [C.c_void_p] * 3 + [C.c_int] * 2 + [C.POINTER(QWeightC)] + [C.c_int] * 2 + [C.POINTER(C.c_int)]
assert reserve(ctx.h) != 0, "the workspace was there"
parts = C.c_int(-1)
status = resid(ctx.h, outs[1].ptr, rows[1].ptr, K, M, C.byref(qw.c), K, N, C.byref(parts))
assert (status, parts.value) == (0, 0), (status, parts.value, lib.awq_last_error())
want, got = (o.download(np.uint16).view(np.float16).astype(np.float64) for o in outs)
assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
print("same product")
"""


def test_residual_product_without_a_split_workspace(tmp_path):
    """900 rows by 4096 columns would leave parts of K to the norm, but need not: where their workspace cannot be had, the
    product runs unsplit, and the failed allocation is not taken for a failed launch."""
    (tmp_path / "no_workspace.c").write_text(NO_WORKSPACE)
    shim = str(tmp_path / "no_workspace.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", shim, str(tmp_path / "no_workspace.c"), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", WITHOUT_WORKSPACE, shim], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "same product" in r.stdout, r.stdout + r.stderr
