"""The batched causal attention at the edges of its tiles, for every head size and every split of queries and keys that the
dispatch knows, through a prefill of two-layer models: the second layer's cache rows depend on the first layer's attention
at every position.  Reference: the same prompt token by token, on the CPU oracle for short prompts, on the GPU's
matrix-vector path (which other tests hold against the oracle) for long ones.  Bar: rel-L2 1e-2 as for every prefill test
(fp16 activations between layers; measured 2e-4 for the attention alone against fp64)."""
import numpy as np
import pytest

import llama_cu_awq_amd as A
from llama_cu_awq_amd import synth
from oracle import oracle
from tests.helpers import f16, rel_l2

pytestmark = pytest.mark.gpu

H64 = dict(dim=256, hidden_dim=256, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=512, seq_len=1280, rope_theta=10000.0)
H128 = dict(dim=384, hidden_dim=256, n_layers=2, n_heads=3, n_kv_heads=1, vocab_size=512, seq_len=1280, rope_theta=10000.0)
H256 = dict(dim=512, hidden_dim=256, n_layers=2, n_heads=2, n_kv_heads=1, vocab_size=512, seq_len=1280, rope_theta=10000.0)
# enough heads for the form that serves 128 queries per workgroup
H128_WIDE = dict(dim=4096, hidden_dim=256, n_layers=2, n_heads=32, n_kv_heads=8, vocab_size=512, seq_len=2304, rope_theta=10000.0)


def _rows(t, cfg, n):
    kv_dim = cfg["dim"] * cfg["n_kv_heads"] // cfg["n_heads"]
    size = cfg["n_layers"] * cfg["seq_len"] * kv_dim
    return [f16(t.download(name, size)).reshape(cfg["n_layers"], cfg["seq_len"], kv_dim)[:, :n] for name in ("key_cache", "value_cache")]


def _prefill(ctx, img, cfg, prompt, parts):
    t = A.Transformer(ctx, image=img)
    t.reset(prompt)
    for i, n in enumerate(parts):
        t.prefill(n, gen_token=(i == len(parts) - 1))
    ctx.sync()
    out = _rows(t, cfg, len(prompt)), f16(t.download("logits", cfg["vocab_size"]))
    t.close()
    return out


def _compare(got, want):
    for a, b in zip(got[0], want[0]):
        for l in range(a.shape[0]):
            assert rel_l2(a[l], b[l]) <= 1e-2, l
            # the last rows on their own: the ends of tiles
            assert rel_l2(a[l][-3:], b[l][-3:]) <= 1e-2, l
    assert rel_l2(got[1], want[1]) <= 1e-2


@pytest.mark.parametrize("parts", [(1,), (31,), (33,), (64,), (65,), (127, 2), (129,), (64, 64)], ids=str)
@pytest.mark.parametrize("cfg", [H64, H128, H256], ids=["heads-of-64", "heads-of-128", "heads-of-256"])
def test_tile_edges_against_the_oracle(ctx, cfg, parts):
    n = sum(parts)
    img = synth.make_model_image(cfg, seed=41, scale_mult=0.5)
    prompt = synth.prompt_tokens(41, n, cfg["vocab_size"])
    o = oracle.Model(img)
    o.reset(prompt)
    for i in range(n):
        o.forward(i >= n - 1)
    kv_dim = cfg["dim"] * cfg["n_kv_heads"] // cfg["n_heads"]
    size = cfg["n_layers"] * cfg["seq_len"] * kv_dim
    rows = [f16(o.buffer(name, size)).reshape(cfg["n_layers"], cfg["seq_len"], kv_dim)[:, :n].copy() for name in ("key_cache", "value_cache")]
    want = rows, f16(o.buffer("logits", cfg["vocab_size"])).copy()
    o.close()
    _compare(_prefill(ctx, img, cfg, prompt, parts), want)


@pytest.mark.parametrize("cfg,parts", [(H64, (511, 1)), (H64, (640, 130)), (H128, (511, 1)), (H128, (500, 12)), (H128, (700, 37, 129)), (H256, (600, 70)),
                                       (H128_WIDE, (1030,)), (H128_WIDE, (1023, 1100))], ids=lambda v: str(v) if isinstance(v, tuple) else f"{v['n_heads']}x{v['dim'] // v['n_heads']}")
def test_long_contexts_against_token_by_token(ctx, cfg, parts):
    n = sum(parts)
    img = synth.make_model_image(cfg, seed=43, scale_mult=0.25)
    prompt = synth.prompt_tokens(43, n, cfg["vocab_size"])
    t = A.Transformer(ctx, image=img)
    t.reset(prompt)
    for i in range(n):
        t.forward(i == n - 1, use_graph=True)
    ctx.sync()
    want = _rows(t, cfg, n), f16(t.download("logits", cfg["vocab_size"]))
    t.close()
    _compare(_prefill(ctx, img, cfg, prompt, parts), want)
