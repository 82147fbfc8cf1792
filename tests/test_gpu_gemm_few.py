"""The few-row form of the batched int4 GEMM (prefills of up to 128 rows): activations in fragment order, K shared by the waves of a
workgroup and by workgroups, against 64-bit products and against the token-by-token path."""
import ctypes as C

import numpy as np
import pytest

import llama_cu_awq_amd as A
from llama_cu_awq_amd import synth
from llama_cu_awq_amd._lib import QWeightC, lib
from tests.helpers import f16, rel_l2

pytestmark = pytest.mark.gpu


class _Plan(C.Structure):  # 32-row units a workgroup, parts of K, the time expected
    _fields_ = [("units", C.c_int), ("parts", C.c_int), ("us", C.c_float)]


_plan = lib["_Z17awq_plan_gemm_fewiiiib"]  # compute units, rows, K, columns, may split
_plan.argtypes, _plan.restype = [C.c_int] * 4 + [C.c_bool], _Plan
_resid = lib["_Z25awq_launch_gemm_few_residP7awq_ctxPtPKtiPK11awq_qweightiiPi"]
_resid.argtypes = [C.c_void_p] * 3 + [C.c_int] + [C.POINTER(QWeightC)] + [C.c_int] * 2 + [C.POINTER(C.c_int)]
_norm_parts = lib["_Z24awq_launch_rmsnorm_partsP7awq_ctxPtS1_PKtiiii"]
_norm_parts.argtypes = [C.c_void_p] * 4 + [C.c_int] * 4
_qkv = lib["_Z19awq_launch_gemm_qkvP7awq_ctxPtS1_S1_PKtiiPK11awq_qweightS6_S6_iiiiPK15HIP_vector_typeIfLj2EEfibb"]
_qkv.argtypes = [C.c_void_p] * 5 + [C.c_int] * 2 + [C.POINTER(QWeightC)] * 3 + [C.c_int] * 4 + [C.c_void_p, C.c_float, C.c_int, C.c_bool, C.c_bool]
_ffn = lib["_Z19awq_launch_gemm_ffnP7awq_ctxPtPKtiiPK11awq_qweightS6_iibbb"]
_ffn.argtypes = [C.c_void_p] * 3 + [C.c_int] * 2 + [C.POINTER(QWeightC)] * 2 + [C.c_int] * 2 + [C.c_bool] * 3
_takes_few = lib["_Z21awq_prefill_takes_fewP7awq_ctxiiii"]
_takes_few.argtypes, _takes_few.restype = [C.c_void_p] + [C.c_int] * 4, C.c_bool


def _fragments(a):
    """[rows][K] in the order of gemm_tile.hpp's fragment_offset, each 8 columns as a packed dword unpacks; what no row fills is
    not a number."""
    M, K = a.shape
    tiles = (M + 31) // 32
    out = np.full((K // 128, 8, tiles, 2, 32, 8), np.nan, np.float16)
    r, c = np.meshgrid(np.arange(M), np.arange(0, K, 8), indexing="ij")
    f = ((c >> 6) & 1) * 4 + ((c >> 3) & 3)
    out[c >> 7, f, r >> 5, (c >> 5) & 1, r & 31] = a.reshape(M, K // 8, 8)[:, :, [0, 4, 1, 5, 2, 6, 3, 7]]
    return out.reshape(-1)


def _from_fragments(bits, M, K):
    """The rows of a block in that order, and whether what no row fills is as it was (all ones)."""
    b = bits.reshape(K // 128, 8, -1, 2, 32, 8).copy()
    r, c = np.meshgrid(np.arange(M), np.arange(0, K, 8), indexing="ij")
    at = (c >> 7, ((c >> 6) & 1) * 4 + ((c >> 3) & 3), r >> 5, (c >> 5) & 1, r & 31)
    rows = b[at][:, :, [0, 2, 4, 6, 1, 3, 5, 7]].reshape(M, K)
    b[at] = 0xFFFF
    return f16(rows), bool((b == 0xFFFF).all())


def _matrix(ctx, key, K, N):
    """On the device, and as the kernels multiply it."""
    w, z, s = synth.make_qweight(key, K, N)
    return A.QWeight.upload(ctx, w, z, s), synth.dequantize(w, z, s, K).astype(np.float32).astype(np.float16).astype(np.float64)


# (rows, K, columns): edges of the row tiles; fewer groups than waves, one group more or less than a multiple of the waves, groups
# that end in the middle of the four or eight that scales and zeros come in; a column tile that the last workgroup fills in part
SHAPES = [(1, 256, 128), (31, 384, 256), (32, 1024, 2048), (33, 1152, 384), (37, 4096, 4096), (64, 896, 1280), (63, 2176, 640),
          (5, 11008, 4096), (33, 11008, 4096), (64, 5248, 5120), (17, 4096, 24576), (48, 1024, 24576), (64, 8192, 16512),
          (65, 384, 256), (96, 4096, 4096), (77, 1152, 12288), (95, 2176, 22016), (65, 11008, 4096), (97, 384, 256), (128, 4096, 4096),
          (127, 1152, 12288), (98, 11008, 4096)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_residual_product_against_fp64(ctx, M, K, N):
    """fp16 weights and activations, fp32 sums, one rounding: apart from that rounding (2.1e-4 in the norm) sums differ by 1e-6.
    Parts of K are added to x by the norm, one rounding too."""
    key = synth.stream_key(61, M, K, N)
    w, z, s = synth.make_qweight(key, K, N)
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K)
    x = synth.normal_f16(synth.stream_key(key, "x"), M * N)
    qw = A.QWeight.upload(ctx, w, z, s)
    dense = synth.dequantize(w, z, s, K).astype(np.float32).astype(np.float16)
    da, dx, do, left = ctx.upload(_fragments(a).view(np.uint16)), ctx.upload(x), ctx.zeros(M * N * 2), C.c_int(-1)
    assert _resid(ctx.h, dx.ptr, da.ptr, M, C.byref(qw.c), K, N, C.byref(left)) == 0
    plan = _plan(256, M, K, N, True)
    assert left.value == (0 if plan.parts == 1 else plan.parts)
    if left.value:
        norm = ctx.upload(synth.normal_f16(synth.stream_key(key, "n"), N, 1.0, 0.02))
        assert _norm_parts(ctx.h, do.ptr, dx.ptr, norm.ptr, N, M, 0, left.value) == 0
    got = f16(dx.download(np.uint16)).reshape(M, N).astype(np.float64)
    want = a.astype(np.float64) @ dense.astype(np.float64).T + x.astype(np.float64).reshape(M, N)
    assert rel_l2(got, want) <= 4e-4
    for at in (np.s_[-1], np.s_[0], np.s_[:, -8:], np.s_[:, :8]):
        assert rel_l2(got[at], want[at]) <= 1e-3


ROWS = (31, 32, 33, 64, 77, 97, 128)
# (K, query columns, key and value columns, head size): the last ones make workgroups of three units that the borders between the
# matrices run through (400, 64 and 208 units of 32)
QKV = [(256, 512, 128, 64), (1152, 1024, 256, 256), (384, 6144, 1280, 128), (384, 12800, 2048, 64), (256, 6656, 6656, 128), (256, 12800, 2048, 256)]
FFN = [(1152, 256), (384, 4352), (256, 8448)]


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("K,Nq,Nkv,head", QKV)
def test_qkv_against_fp64(ctx, M, K, Nq, Nkv, head):
    """Rotated q and k, v as it is, cache rows from a position on.  q and k are rounded to fp16 before the rotation and behind it, v once
    (2.1e-4 in the norm each, 3.0e-4 together)."""
    key, pos0 = synth.stream_key(64, M, K, Nq), 5
    mats = [_matrix(ctx, synth.stream_key(key, name), K, n) for name, n in (("q", Nq), ("k", Nkv), ("v", Nkv))]
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K)
    angle = np.random.default_rng(M + Nq).uniform(0, 2 * np.pi, (pos0 + M, head // 2))
    rope = np.stack([np.cos(angle), np.sin(angle)], axis=-1).astype(np.float32)
    da, dr, outs = ctx.upload(_fragments(a).view(np.uint16)), ctx.upload(rope), []
    for n, first in ((Nq, 0), (Nkv, pos0), (Nkv, pos0)):
        outs.append((ctx.upload(np.full((first + M + 1) * n, 0xFFFF, np.uint16)), first, n))
    assert _qkv(ctx.h, *(o.ptr for o, _, _ in outs), da.ptr, K, M, *(C.byref(m.c) for m, _ in mats), K, Nq, Nkv, head, dr.ptr, 10000.0, pos0, True, True) == 0
    for i, (out, first, n) in enumerate(outs):
        bits = out.download(np.uint16).reshape(-1, n)
        assert (bits[:first] == 0xFFFF).all() and (bits[first + M :] == 0xFFFF).all()
        want = a.astype(np.float64) @ mats[i][1].T
        if i < 2:
            x, y = (want.reshape(M, -1, 2, head // 2)[:, :, j] for j in (0, 1))
            c, s = (rope[pos0:, None, :, j].astype(np.float64) for j in (0, 1))
            want = np.stack([x * c - y * s, x * s + y * c], axis=2).reshape(M, n)
        got = f16(bits[first : first + M]).astype(np.float64)
        assert rel_l2(got, want) <= 4e-4
        for at in (np.s_[-1], np.s_[0], np.s_[:, -32:], np.s_[:, :32]):
            assert rel_l2(got[at], want[at]) <= 1e-3


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("K,N", FFN)
def test_gate_and_up_against_fp64(ctx, M, K, N):
    """silu(gate) * up in fp32, rounded once, in fragment order; what lies between the last row and the end of its tile is not written."""
    key = synth.stream_key(65, M, K, N)
    (gate, gate64), (up, up64) = (_matrix(ctx, synth.stream_key(key, name), K, N) for name in ("gate", "up"))
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K)
    da, dh = ctx.upload(_fragments(a).view(np.uint16)), ctx.upload(np.full((M + 31) // 32 * 32 * N, 0xFFFF, np.uint16))
    assert _ffn(ctx.h, dh.ptr, da.ptr, K, M, C.byref(gate.c), C.byref(up.c), K, N, True, True, True) == 0
    got, rest = _from_fragments(dh.download(np.uint16), M, N)
    g, u = (a.astype(np.float64) @ m.T for m in (gate64, up64))
    want = g / (1 + np.exp(-g)) * u
    assert rest and rel_l2(got, want) <= 4e-4
    for at in (np.s_[-1], np.s_[0], np.s_[:, -32:], np.s_[:, :32]):
        assert rel_l2(got[at], want[at]) <= 1e-3


def test_every_form_is_taken():
    """In each of the three kernels that a form has: the single-matrix one, QKV and gate/up (these do not split K)."""
    forms = {(m, u) for m in (1, 2, 3, 4) for u in (1, 2, 3)} - {(4, 3)}
    tiles = lambda M: (M + 31) // 32
    taken = {(tiles(M), p.units, p.parts > 1) for M, K, N in SHAPES for p in [_plan(256, M, K, N, True)]}
    assert {t[:2] for t in taken} == forms
    assert {t[0] for t in taken if t[2]} == {1, 2, 3, 4}
    qkv = {(shape, M): _plan(256, M, shape[0], shape[1] + 2 * shape[2], False).units for shape in QKV for M in ROWS}
    assert {(tiles(M), u) for (_, M), u in qkv.items()} == forms
    # a unit of q and one of k in one workgroup, one of k and one of v
    border = {(tiles(M), u) for (shape, M), u in qkv.items() if shape[1] // 32 % u and (shape[1] + shape[2]) // 32 % u}
    assert border == {(1, 3), (2, 3), (3, 3)}
    assert {(tiles(M), _plan(256, M, K, 2 * N, False).units) for K, N in FFN for M in ROWS} == forms


def test_infinite_activation_stays_in_its_row(ctx):
    M, K, N = 40, 1152, 384
    key = synth.stream_key(62, M, K, N)
    qw = A.QWeight.upload(ctx, *synth.make_qweight(key, K, N))
    a = synth.normal_f16(synth.stream_key(key, "a"), M * K).reshape(M, K).copy()
    a[39, K - 1] = np.inf  # the row that rows past the last read in its place
    da, dx, left = ctx.upload(_fragments(a).view(np.uint16)), ctx.zeros(M * N * 2), C.c_int(-1)
    assert _resid(ctx.h, dx.ptr, da.ptr, M, C.byref(qw.c), K, N, C.byref(left)) == 0 and left.value == 0
    got = f16(dx.download(np.uint16)).reshape(M, N)
    assert np.isfinite(got[:39]).all() and not np.isfinite(got[39]).all()


MODELS = {"64": dict(dim=512, hidden_dim=1408, n_heads=8, n_kv_heads=2), "128": dict(dim=1024, hidden_dim=2816, n_heads=8, n_kv_heads=8),
          "256": dict(dim=1536, hidden_dim=2048, n_heads=6, n_kv_heads=1), "wide": dict(dim=4096, hidden_dim=11008, n_heads=32, n_kv_heads=32),
          "64 wide": dict(dim=2048, hidden_dim=5632, n_heads=32, n_kv_heads=4)}


@pytest.mark.parametrize("model", MODELS)
def test_prefill_against_token_by_token(ctx, model):
    """Passes at the edges of the row tiles, one behind another (the attention takes its forms for few and for many keys): cache rows
    and logits of the token-by-token path within the tolerance of the batched one."""
    m = MODELS[model]
    cfg = dict(m, n_layers=2, vocab_size=512, seq_len=1024, rope_theta=10000.0)
    kv_dim = m["dim"] * m["n_kv_heads"] // m["n_heads"]
    parts = (1, 31, 32, 33, 63, 64, 300, 40, 5, 65, 96, 97, 128)
    n = sum(parts)
    assert all(_takes_few(ctx.h, p, m["dim"], kv_dim, m["hidden_dim"]) for p in parts if p <= 64)
    assert all(_takes_few(ctx.h, p, m["dim"], kv_dim, m["hidden_dim"]) == ("wide" in model) for p in (65, 96, 97, 128))
    assert not _takes_few(ctx.h, 129, m["dim"], kv_dim, m["hidden_dim"])
    img = synth.make_model_image(cfg, seed=63, scale_mult=0.25)
    prompt = synth.prompt_tokens(63, n, cfg["vocab_size"])
    t = A.Transformer(ctx, image=img)
    size = 2 * cfg["seq_len"] * kv_dim

    def state():
        ctx.sync()
        rows = [f16(t.download(name, size)).reshape(2, cfg["seq_len"], kv_dim)[:, :n].copy() for name in ("key_cache", "value_cache")]
        return rows, f16(t.download("logits", cfg["vocab_size"])).copy()

    t.reset(prompt)
    for i in range(n):
        t.forward(i == n - 1, use_graph=True)
    want, want_logits = state()
    t.reset(prompt)
    for i, p in enumerate(parts):
        t.prefill(p, gen_token=i == len(parts) - 1)
    got, logits = state()
    t.close()
    for a, b in zip(got, want):
        at = 0
        for p in parts:
            for l in range(2):
                assert rel_l2(a[l, at : at + p], b[l, at : at + p]) <= 1e-2, (p, l)
                assert rel_l2(a[l, at + p - 1], b[l, at + p - 1]) <= 2e-2, (p, l)
            at += p
    assert rel_l2(logits, want_logits) <= 1e-2
