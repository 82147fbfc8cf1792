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


# ---------------------------------------------------------------- scores by design
def _designed(cfg, seed, reach, offset=0.0):
    """A model whose first layer's scores are known: a query's is `reach` times the key token's level, -1 .. 1 in 65 steps
    (token v has level (v % 65) / 32 - 1), plus `offset`, at every distance (the only pair of dimensions in use turns least)."""
    dim, hid, heads, kv, vocab = (cfg[k] for k in ("dim", "hidden_dim", "n_heads", "n_kv_heads", "vocab_size"))
    hs = dim // heads
    img = synth.make_model_image(cfg, seed=seed, scale_mult=0.25)
    rng = np.random.default_rng(seed)
    # columns 0 .. 127 of every embedding are 1, of the next 128 as many are +1 as the level says, the others +-1 in pairs
    embed = img[32 : 32 + 2 * vocab * dim].view(np.float16).reshape(vocab, dim)
    embed[:, :128] = 1
    for v in range(vocab):
        ups = 2 * (v % 65)  # of 128
        embed[v, 128:256] = rng.permutation(np.repeat([1.0, -1.0], [ups, 128 - ups]))
        embed[v, 256:] = rng.choice([-1.0, 1.0], dim - 256)
    off = 32 + 4 * vocab * dim + 2 * dim

    def matrix(K, N):
        nonlocal off
        pwh, pzh, sh = synth.strides(K)
        parts = []
        for width, dtype in ((pwh, np.uint32), (pzh, np.uint32), (sh, np.float16)):
            n = N * width * np.dtype(dtype).itemsize
            parts.append(img[off : off + n].view(dtype).reshape(N, width))
            off += n
        return parts

    def functional(m, rows, first, scale):
        """`rows` of a matrix become scale times the sum over 128 columns."""
        w, z, s = m
        w[rows], z[rows], s[rows] = 0, 0, scale
        w[rows, first // 8 : first // 8 + 16] = 0x11111111

    alpha = hs**-0.5
    q, k = matrix(dim, dim), matrix(dim, kv * hs)
    matrix(dim, kv * hs)
    for m in (q, k):
        m[0][:], m[1][:] = 0, 0
    functional(q, np.arange(heads) * hs + hs // 2 - 1, 0, 1 / 128)  # 1 for every token
    k_rows = np.arange(kv) * hs + hs // 2 - 1
    functional(k, k_rows, 128, reach / alpha / 128)
    k[0][k_rows, :16], k[2][k_rows, 0] = 0x11111111, offset / alpha / 128
    matrix(dim, dim)
    for K, N in ((dim, hid), (dim, hid), (hid, dim)):
        matrix(K, N)
    img[off : off + 2 * dim].view(np.float16)[:] = 1  # the first norm's weights
    return img


def _token(level, rng, vocab):
    """A token of the level nearest to `level`."""
    v = int(np.clip(np.round((level + 1) * 32), 0, 64))
    return int(v + 65 * rng.integers(0, vocab // 65))


def _token_by_token(ctx, img, cfg, prompt):
    t = A.Transformer(ctx, image=img)
    t.reset(prompt)
    for i in range(len(prompt)):
        t.forward(i == len(prompt) - 1, use_graph=True)
    ctx.sync()
    out = _rows(t, cfg, len(prompt)), f16(t.download("logits", cfg["vocab_size"]))
    t.close()
    return out


def _oracle(img, cfg, prompt):
    o = oracle.Model(img)
    o.reset(prompt)
    for i in range(len(prompt)):
        o.forward(i >= len(prompt) - 1)
    kv_dim = cfg["dim"] * cfg["n_kv_heads"] // cfg["n_heads"]
    size = cfg["n_layers"] * cfg["seq_len"] * kv_dim
    rows = [f16(o.buffer(name, size)).reshape(cfg["n_layers"], cfg["seq_len"], kv_dim)[:, : len(prompt)].copy() for name in ("key_cache", "value_cache")]
    out = rows, f16(o.buffer("logits", cfg["vocab_size"])).copy()
    o.close()
    return out


# one profile of scores over the positions: the maximum grows by more than the rescale's threshold again and again; stands in the
# first tile; differs by 40 and more between the key slices of a tile
PROFILES = {
    "ascending": lambda i, n: 2 * i / n - 1,
    "descending": lambda i, n: 1 - 2 * i / n,
    "by-slice": lambda i, n: (-0.7, 0.1, 0.9, 0.4)[(i // 32) % 4] + 0.05 * (i % 3),
}
# every form of the dispatch: (heads, prompt): one tile, 64 queries by 2 slices, 32 queries by 4 slices, 128 queries
FORMS = [(H64, (64,)), (H64, (300,)), (H64, (600, 40)), (H128, (64,)), (H128, (300,)), (H128, (600, 40)), (H256, (64,)), (H256, (300,)), (H256, (600, 40)),
         (H128_WIDE, (1030,))]
FORM_IDS = [f"{c['n_heads']}x{c['dim'] // c['n_heads']}-{'+'.join(map(str, p))}" for c, p in FORMS]


@pytest.mark.parametrize("profile", PROFILES)
@pytest.mark.parametrize("cfg,parts", FORMS, ids=FORM_IDS)
def test_maxima_that_move(ctx, cfg, parts, profile):
    """Scores from -60 to 60 in known order, so that single keys carry the result.  One product makes a score, so both sides
    round the same one; what differs is rounded to fp16 five times on the way to the second layer's rows (p, the output, the
    residual, the norm, the product: 2^-11 / sqrt(3) each, 6e-4 together): 3e-3."""
    n = sum(parts)
    img = _designed(cfg, 61, 60.0)
    rng = np.random.default_rng(62)
    prompt = [_token(PROFILES[profile](i, n), rng, cfg["vocab_size"]) for i in range(n)]
    want = _token_by_token(ctx, img, cfg, prompt) if cfg is H128_WIDE else _oracle(img, cfg, prompt)
    got = _prefill(ctx, img, cfg, prompt, parts)
    for a, b in zip(got[0], want[0]):
        assert rel_l2(a[1], b[1]) <= 3e-3
        for at in range(0, n, 32):
            assert rel_l2(a[1][at : at + 32], b[1][at : at + 32]) <= 3e-3, at
    assert rel_l2(got[1], want[1]) <= 1e-2


@pytest.mark.parametrize("cfg,parts", [(H64, (64,)), (H64, (100,)), (H256, (100,))], ids=["64x1", "64x2", "256"])
def test_scores_far_below_zero(ctx, cfg, parts):
    """A constant added to every score changes no softmax: scores of -166 .. -134, whose exponentials are zero in fp32, against
    -16 .. 16.  Both are multiples of a half, which fp16 holds; over 100 positions the pair turns by 0.0133, and what the fp16
    factors keep of that, 0.0133^2 of a score, is below the rounding of the far ones (0.03 of 0.06) and moves the near ones by
    up to 16 x 0.0133^2 = 0.003, a probability by 3e-3.  With the five fp16 roundings of the test above (6e-4): 4e-3."""
    prompt = [_token(PROFILES["by-slice"](i, sum(parts)), np.random.default_rng(64 + i), cfg["vocab_size"]) for i in range(sum(parts))]
    near, far = (_prefill(ctx, _designed(cfg, 65, 16.0, offset), cfg, prompt, parts) for offset in (0.0, -150.0))
    for a, b in ((near[0][0][1], far[0][0][1]), (near[0][1][1], far[0][1][1]), (near[1], far[1])):
        assert np.isfinite(b).all() and rel_l2(a, b) <= 4e-3


@pytest.mark.parametrize("cfg,parts", FORMS, ids=FORM_IDS)
def test_infinite_values_stay_with_the_queries_that_see_them(ctx, cfg, parts):
    """One token's value row overflows to infinity; the rows of the tokens before it are those of the prompt without it."""
    n, vocab, dim = sum(parts), cfg["vocab_size"], cfg["dim"]
    at = n - parts[-1] // 3 - 1  # of the last call, in the middle of a block of queries
    img = synth.make_model_image(cfg, seed=63, scale_mult=0.5)
    embed = img[32 : 32 + 2 * vocab * dim].view(np.float16).reshape(vocab, dim)
    embed[:] = np.sign(embed) + (embed == 0)
    embed[:, 0] = 0
    embed[vocab - 1, 0] = 4
    # row 0 of the first layer's values: 60000 times column 0
    off = 32 + 4 * vocab * dim + 2 * dim
    kv_dim = dim * cfg["n_kv_heads"] // cfg["n_heads"]
    pwh, pzh, sh = synth.strides(dim)
    off += (dim + kv_dim) * (4 * pwh + 4 * pzh + 2 * sh)
    w, z, s = off, off + 4 * kv_dim * pwh, off + 4 * kv_dim * (pwh + pzh)
    img[w : w + 4 * pwh].view(np.uint32)[:] = [0xF] + [0] * (pwh - 1)
    img[z : z + 4 * pzh].view(np.uint32)[:] = 0
    img[s : s + 2 * sh].view(np.float16)[:] = 4000
    prompt = [int(v) % (vocab - 1) for v in synth.prompt_tokens(63, n, vocab)]
    want = _prefill(ctx, img, cfg, prompt, parts)[0]
    prompt[at] = vocab - 1
    got = _prefill(ctx, img, cfg, prompt, parts)[0]
    assert np.isposinf(got[1][0, at, 0]) and np.isfinite(got[1][0]).sum() == got[1][0].size - 1
    for a, b in zip(got, want):
        assert rel_l2(a[1, :at], b[1, :at]) <= 1e-3  # (the tokens before are the same ones; only the order of sums may differ)
        assert not np.isfinite(a[1, at:]).all(axis=1).any()
