"""The work that users of this framework have it do, as cases whose speed and results can be compared between versions.

A case is one pass of a user's program through the public entry points (`llama_cu_awq_amd`): a sampled or greedy decode, a
batched prefill of a prompt, or a launcher-level product.  Models are built on the GPU from the seed alone, in the packed
file's layout, with the benchmark's distributions (4-bit weights and zero points uniform, scales uniform) and two changes
that let results be compared at all:

 * The scale range is an eighth of the benchmark's, so that the residual stream of a deep model keeps to the range of fp16
   and its outputs do not turn on single rounding errors.
 * Embeddings are N(0, 1) and a row of the classifier is partly the embedding of another token, so that the next token leads
   by a margin, as it mostly does in a trained model: a decode of several tokens then follows the same path however its sums
   are rounded.
"""
import math

import numpy as np
import torch

import llama_cu_awq_amd as A
from llama_cu_awq_amd import synth

SCALE_MULT = 0.125
LEAD = 0.2  # share of a classifier row that is another token's embedding


def _model(base, **changes):
    """The plain fields of a model configuration, for a case."""
    return {**{k: v for k, v in base.items() if k != "rope_theta"}, **changes}


def _vec(name, **sizes):
    return {"name": name, "kind": "mlp_vec", **sizes}


def listed():
    small = dict(dim=2048, hidden_dim=5632, n_layers=22, n_heads=32, n_kv_heads=4, vocab_size=32000, seq_len=2048)
    grouped = dict(dim=4096, hidden_dim=14336, n_layers=16, n_heads=32, n_kv_heads=8, vocab_size=128256, seq_len=2048)
    slice_70b = _model(synth.CONFIG_70B, n_layers=8)
    slice_13b = _model(synth.CONFIG_13B, n_layers=20)
    c7 = _model(synth.CONFIG_7B)
    return [
        # one token's feed-forward block through the launchers, as the reference's host code calls them: the smallest calls
        _vec("mlp_vec_4096", K=4096, H=11008),
        # a batch of rows that is no multiple of any tile, as a serving loop collects it
        {"name": "gemm_rows_77", "kind": "gemm", "M": 77, "K": 5120, "N": 13824},
        # the reference's headline use: greedy decode of one sequence from the start, the graph replayed per token
        {"name": "decode_7b", "kind": "decode", **c7, "start": 0, "steps": 16},
        # late in a conversation: the cache is as large a part of the traffic as it gets (half the layers of the 13B shape)
        {"name": "decode_13b_late", "kind": "decode", **slice_13b, "start": 1536, "steps": 12},
        # grouped queries, the largest matrices (a tenth of the 70B shape's layers)
        {"name": "decode_70b_slice", "kind": "decode", **slice_70b, "start": 300, "steps": 12},
        # a small model on a large chip, 64-wide heads: launches and latencies
        {"name": "decode_small", "kind": "decode", **small, "start": 40, "steps": 24},
        # the command line's default sampler (temperature 0.5, top-p 0.6) at a large vocabulary
        {"name": "sample_grouped", "kind": "sample", **grouped, "start": 200, "steps": 12},
        # a question of a few dozen tokens
        {"name": "prefill_7b_37", "kind": "prefill", **c7, "first": 37, "second": 0},
        # the benchmark's prompt
        {"name": "prefill_7b_512", "kind": "prefill", **c7, "first": 512, "second": 0},
        # a document that nearly fills the context
        {"name": "prefill_7b_2000", "kind": "prefill", **c7, "first": 2000, "second": 0},
        # a prompt and, behind it, a second message, on the largest matrices
        {"name": "prefill_70b_two", "kind": "prefill", **slice_70b, "first": 650, "second": 150},
        # 64-wide heads
        {"name": "prefill_small_700", "kind": "prefill", **small, "first": 700, "second": 0},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` from lo to hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def _drawn_model(rng, step):
    """A model of a few layers whose sizes are multiples of `step`."""
    head = rng.choice((64, 128, 128))
    kv = rng.choice((1, 2, 4, 5, 8, 8))
    mul = rng.choice((1, 1, 2, 4, 8))
    heads = kv * mul
    while heads * head < 1024 or heads * head > 8192 or (kv * head) % step or (heads * head) % step:
        kv = rng.choice((2, 4, 5, 8, 10, 16, 26, 32, 40))
        mul = rng.choice((1, 1, 2, 4, 8))
        heads = kv * mul
    dim = heads * head
    hidden = _log(rng, 2 * dim, min(28672, 4 * dim), step)
    layers = max(1, min(rng.randint(3, 10), int(5e9 / (4 * dim * dim + 3 * dim * hidden))))
    return dict(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=heads, n_kv_heads=kv,
                vocab_size=_log(rng, 8000, 128256, 8), seq_len=2048)


def draw(rng):
    kind = rng.choice(("mlp_vec", "gemm", "decode", "decode", "sample", "prefill", "prefill", "prefill"))
    if kind == "mlp_vec":
        return {"kind": kind, "K": _log(rng, 512, 8192, 8), "H": _log(rng, 2048, 28672, 8)}
    if kind == "gemm":
        return {"kind": kind, "M": _log(rng, 1, 2048), "K": _log(rng, 1024, 14336, 32), "N": _log(rng, 1024, 28672, 128)}
    if kind in ("decode", "sample"):
        start = 0 if rng.random() < 0.2 else _log(rng, 8, 2000)
        return {"kind": kind, **_drawn_model(rng, 32), "start": start, "steps": rng.randint(6, 24)}
    first = _log(rng, 4, 2040)
    second = 0 if rng.random() < 0.6 or first > 1900 else _log(rng, 1, 2040 - first)
    return {"kind": kind, **_drawn_model(rng, 128), "first": first, "second": second}


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1 + int(seed))
    return g


def _put_matrix(image, off, K, N, g, scale_mult=SCALE_MULT):
    """A random packed matrix of N rows over K inputs into `image` (bytes on the GPU) from `off` on; the end of it."""
    pwh, pzh, sh = synth.strides(K)
    w = image[off : off + N * pwh * 4].view(torch.int32)
    w.random_(-(1 << 31), (1 << 31) - 1, generator=g)
    if K % 32:  # nibbles past K are zero
        last = w.view(N, pwh)[:, K // 8 :]
        last.zero_()
    off += N * pwh * 4
    z = image[off : off + N * pzh * 4].view(torch.int32).view(N, pzh)
    z.random_(-(1 << 31), (1 << 31) - 1, generator=g)
    if sh % 8:
        z[:, -1] &= (1 << (4 * (sh % 8))) - 1
    off += N * pzh * 4
    s = image[off : off + N * sh * 2].view(torch.float16)
    s.copy_(torch.rand(N * sh, device="cuda", generator=g).mul_(0.018 * scale_mult).add_(0.002 * scale_mult))
    return off + N * sh * 2


def _image(cfg, g):
    """A whole model in the packed file's order, as bytes on the host."""
    dim, hid, vocab = cfg["dim"], cfg["hidden_dim"], cfg["vocab_size"]
    kv_dim = dim * cfg["n_kv_heads"] // cfg["n_heads"]
    image = torch.empty(synth.model_bytes(cfg), dtype=torch.uint8, device="cuda")
    head = np.array([dim, hid, cfg["n_layers"], cfg["n_heads"], cfg["n_kv_heads"], vocab, cfg["seq_len"]], np.int32)
    head = np.concatenate([head.view(np.uint8), np.array([10000.0], np.float32).view(np.uint8)])
    image[:32] = torch.from_numpy(head).cuda()
    off = 32

    def dense(n):
        nonlocal off
        off += 2 * n
        return image[off - 2 * n : off].view(torch.float16)

    embed = dense(vocab * dim).view(vocab, dim)
    embed.normal_(generator=g)
    wcls = dense(vocab * dim).view(vocab, dim)
    wcls.normal_(generator=g)
    shift = 1 + int(torch.randint(0, vocab - 1, (1,), device="cuda", generator=g))
    wcls.mul_(0.02 * math.sqrt(1 - LEAD * LEAD)).add_(torch.roll(embed, shift, 0), alpha=0.02 * LEAD)
    dense(dim).copy_(1 + 0.02 * torch.randn(dim, device="cuda", generator=g))
    for _ in range(cfg["n_layers"]):
        for K, N in ((dim, dim), (dim, kv_dim), (dim, kv_dim), (dim, dim), (dim, hid), (dim, hid), (hid, dim)):
            off = _put_matrix(image, off, K, N, g)
        for _ in range(2):
            dense(dim).copy_(1 + 0.02 * torch.randn(dim, device="cuda", generator=g))
    assert off == image.numel()
    return image.cpu().numpy()


class _Model:
    """A loaded model with its context; freed with the last of its users."""

    def __init__(self, image):
        torch.cuda.synchronize()
        self.ctx = A.Context(0)
        self.t = A.Transformer(self.ctx, image=image)

    def __del__(self):
        self.t.close()
        self.ctx.close()


class _View:
    """A part of a model's run state, for torch; keeps the model."""

    def __init__(self, model, name, shape):
        self.model = model
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f2", "data": (int(getattr(model.t.state, name)), False), "version": 2}


def _prepare_model(case, g):
    cfg = {k: case[k] for k in ("dim", "hidden_dim", "n_layers", "n_heads", "n_kv_heads", "vocab_size", "seq_len")}
    m = _Model(_image(cfg, g))
    kv_dim = cfg["dim"] * cfg["n_kv_heads"] // cfg["n_heads"]
    s = {"model": m, "t": m.t, "ctx": m.ctx, "vocab": cfg["vocab_size"], "case": case}
    s["logits"] = torch.as_tensor(_View(m, "logits", (cfg["vocab_size"],)), device="cuda")
    for name in ("key_cache", "value_cache"):
        s[name] = torch.as_tensor(_View(m, name, (cfg["n_layers"], cfg["seq_len"], kv_dim)), device="cuda")
    return s


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("mlp_vec", "gemm"):
        ctx = A.Context(0)
        s = {"ctx": ctx, "case": case}

        def matrix(K, N):
            pwh, pzh, sh = synth.strides(K)
            b = torch.empty(N * (pwh * 4 + pzh * 4 + sh * 2), dtype=torch.uint8, device="cuda")
            _put_matrix(b, 0, K, N, g)
            s.setdefault("keep", []).append(b)
            p = b.data_ptr()
            return A.QWeight(p, p + N * pwh * 4, p + N * (pwh + pzh) * 4)

        if kind == "mlp_vec":
            K, H = case["K"], case["H"]
            s["x"] = torch.randn(K, device="cuda", generator=g).half()
            s["norm"] = (1 + 0.02 * torch.randn(K, device="cuda", generator=g)).half()
            s["gate"], s["up"], s["down"] = matrix(K, H), matrix(K, H), matrix(H, K)
            s["h"] = torch.zeros(H, dtype=torch.float16, device="cuda")
            s["out"] = torch.zeros(K, dtype=torch.float16, device="cuda")
        else:
            M, K, N = case["M"], case["K"], case["N"]
            s["a"] = torch.randn(M, K, device="cuda", generator=g).half()
            s["w"] = matrix(K, N)
            s["out"] = torch.zeros(M, N, dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        return s
    s = _prepare_model(case, g)
    vocab = case["vocab_size"]
    rng = np.random.default_rng(int(seed))
    if kind == "prefill":
        s["prompt"] = rng.integers(3, vocab, case["first"] + case["second"]).tolist()
        return s
    start, steps = case["start"], case["steps"]
    if start:  # what earlier passes left in the cache
        for name in ("key_cache", "value_cache"):
            for layer in s[name]:
                layer[:start].normal_(generator=g)
    torch.cuda.synchronize()
    s["token"] = int(rng.integers(3, vocab))
    # recorded once per model, as the benchmark does before its clock starts
    s["t"].capture(start + steps)
    if kind == "sample":
        s["sampler"] = A.Sampler(s["ctx"], vocab, 0.5, 0.6, 1 + int(seed))
    return s


# ---------------------------------------------------------------- passes
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mlp_vec":
        ctx, K, H = s["ctx"], case["K"], case["H"]
        A.rmsnorm_ffn_matvec_silu(ctx, s["h"].data_ptr(), s["x"].data_ptr(), s["norm"].data_ptr(), s["gate"], s["up"], K, H)
        A.matmul_q(ctx, s["out"].data_ptr(), s["h"].data_ptr(), s["down"], H, K)
        return s["h"], s["out"]
    if kind == "gemm":
        M, K, N = case["M"], case["K"], case["N"]
        A.gemm_q(s["ctx"], s["out"].data_ptr(), N, s["a"].data_ptr(), K, M, s["w"], K, N)
        return s["out"]
    t = s["t"]
    if kind == "prefill":
        t.reset(s["prompt"])
        first, second = case["first"], case["second"]
        t.prefill(first, gen_token=not second)
        if second:
            t.prefill(second)
        n = first + second
        s["ctx"].sync()
        return {"logits": s["logits"], "k": s["key_cache"][:, :n], "v": s["value_cache"][:, :n], "token": np.array([t.token(n)])}
    start, steps = case["start"], case["steps"]
    t.set_pos(start, s["token"])
    tokens = np.empty(steps, np.int64)
    for i in range(steps):
        if kind == "sample":
            t.forward_logits(use_graph=True)
            t.sample(s["sampler"])
        else:
            t.forward(True, use_graph=True)
        s["ctx"].sync()  # each token is there to be printed
        tokens[i] = t.token(start + 1 + i)
    return {"logits": s["logits"], "k": s["key_cache"][:, start : start + steps], "v": s["value_cache"][:, start : start + steps], "tokens": tokens}


# ---------------------------------------------------------------- what a pass cannot do without
def _matrix_bytes(K, N):
    pwh, pzh, sh = synth.strides(K)
    return N * (pwh * 4 + pzh * 4 + sh * 2)


def work(case):
    kind = case["kind"]
    if kind == "mlp_vec":
        K, H = case["K"], case["H"]
        return {"bytes": 2 * _matrix_bytes(K, H) + _matrix_bytes(H, K) + 2 * (3 * K + H), "flops": 6 * K * H}
    if kind == "gemm":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": _matrix_bytes(K, N) + 2 * M * (K + N), "flops": 2 * M * K * N}
    dim, hid, L, vocab = case["dim"], case["hidden_dim"], case["n_layers"], case["vocab_size"]
    kv_dim = dim * case["n_kv_heads"] // case["n_heads"]
    params = L * (2 * dim * dim + 2 * dim * kv_dim + 3 * dim * hid)
    layers = L * (2 * _matrix_bytes(dim, dim) + 2 * _matrix_bytes(dim, kv_dim) + 2 * _matrix_bytes(dim, hid) + _matrix_bytes(hid, dim) + 4 * dim)
    head = 2 * dim * vocab + 2 * vocab + 2 * dim
    if kind == "prefill":
        n, calls = case["first"] + case["second"], 2 if case["second"] else 1
        # each call streams the weights once, embeds its tokens, writes its cache rows and ends in the classifier; the
        # second also reads the first one's cache rows
        moved = calls * (layers + head) + n * 2 * dim + L * kv_dim * 4 * (n + (case["first"] if calls == 2 else 0))
        flops = 2 * n * params + calls * 2 * dim * vocab + L * 2 * dim * n * (n + 1)
        return {"bytes": moved, "flops": flops}
    start, steps = case["start"], case["steps"]
    positions = sum(start + i for i in range(steps))
    moved = steps * (layers + head + 2 * dim) + L * kv_dim * 4 * (positions + steps)
    flops = 2 * steps * (params + dim * vocab) + L * 4 * dim * (positions + steps)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times what two correct evaluations at these precisions are apart.

    Products: results rounded once to fp16 against a product in 64 bits, 2.1e-4 in the norm and 5e-4 at the worst element.
    Models: fp16 activations between layers, a batched prefill (matrix cores) against the same prompt token by token
    (dot products): logits 1.1e-3 to 2.5e-3, cache rows 0.7e-3 to 2.4e-3 in the norm, 1.4e-2 at the worst element.
    """
    if case["kind"] in ("mlp_vec", "gemm"):
        return {"rel": 1e-3, "max": 2e-3}
    return {"rel": 1e-2, "max": 6e-2}
