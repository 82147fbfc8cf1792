"""GPU parity of the whole decode path against the CPU oracle on small models.

Bar (from the benchmark definition): logits within rel-L2 1e-2 of the oracle at every step, greedy tokens
identical for the first 32 steps.  The run state after one token is also compared buffer by buffer.
"""
import numpy as np
import pytest

import llama_cu_awq_amd as A
from llama_cu_awq_amd import synth
from oracle import oracle
from tests.helpers import f16, rel_l2
from tests.test_gpu_prefill_attention import PROFILES, _designed, _rows, _token

pytestmark = pytest.mark.gpu

TINY = dict(dim=256, hidden_dim=768, n_layers=2, n_heads=2, n_kv_heads=2, vocab_size=512, seq_len=64, rope_theta=10000.0)
SMALL = dict(dim=1024, hidden_dim=2752, n_layers=4, n_heads=8, n_kv_heads=8, vocab_size=4096, seq_len=160, rope_theta=10000.0)
GQA = dict(dim=512, hidden_dim=1536, n_layers=2, n_heads=8, n_kv_heads=2, vocab_size=1024, seq_len=64, rope_theta=10000.0)


@pytest.fixture(scope="module", params=["tiny", "small", "gqa"])
def pair(request, ctx):
    cfg = {"tiny": TINY, "small": SMALL, "gqa": GQA}[request.param]
    img = synth.make_model_image(cfg, seed=0)
    t = A.Transformer(ctx, image=img)
    o = oracle.Model(img)
    yield cfg, t, o
    t.close()
    o.close()


def test_header_round_trip(pair):
    cfg, t, o = pair
    for k in ("dim", "hidden_dim", "n_layers", "n_heads", "n_kv_heads", "vocab_size", "seq_len"):
        assert t.config[k] == cfg[k] == o.config[k]


@pytest.mark.parametrize("mode", [A.SCHEDULE_REFERENCE, A.SCHEDULE_FUSED, A.SCHEDULE_PERSISTENT])
def test_one_token_state(pair, mode):
    cfg, t, o = pair
    prompt = synth.prompt_tokens(1, 4, cfg["vocab_size"])
    t.reset(prompt)
    o.reset(prompt)
    for step in range(3):
        t.forward(gen_token=False, use_graph=False, mode=mode)
        o.forward(gen_token=False)
    t.ctx.sync()
    assert t.pos == 3 and o.pos == 3
    assert [t.token(i) for i in range(4)] == prompt == o.tokens(4)  # prompt steps leave the token list alone
    kv_dim = cfg["dim"] * cfg["n_kv_heads"] // cfg["n_heads"]
    for name, n in (("logits", cfg["vocab_size"]), ("hb", cfg["hidden_dim"]), ("q", cfg["dim"]), ("key_cache", 3 * kv_dim), ("value_cache", 3 * kv_dim)):
        got = f16(t.download(name, n))
        want = f16(o.buffer(name, n))
        assert rel_l2(got, want) <= 1e-2, name


@pytest.mark.parametrize("mode,graph", [(A.SCHEDULE_REFERENCE, False), (A.SCHEDULE_FUSED, False), (A.SCHEDULE_FUSED, True), (A.SCHEDULE_REFERENCE, True), (A.SCHEDULE_PERSISTENT, False)])
def test_greedy_decode_matches_oracle(pair, mode, graph):
    cfg, t, o = pair
    n_prompt, steps = 8, min(48, cfg["seq_len"] - 1)
    prompt = synth.prompt_tokens(2, n_prompt, cfg["vocab_size"])
    want_tokens, want_pos, want_logits = o.generate(prompt, steps, ignore_eos=True, want_logits=True)
    got_logits = {}
    got_tokens, got_pos = t.generate(prompt, steps, ignore_eos=True, use_graph=graph, mode=mode, on_logits=lambda p, l: got_logits.__setitem__(p, f16(l)))
    assert got_pos == want_pos == steps
    # prompt tokens are echoed unchanged
    assert got_tokens[:n_prompt] == prompt
    first_diff = next((i for i in range(len(want_tokens)) if got_tokens[i] != want_tokens[i]), None)
    margin = None
    if first_diff is not None:
        l = np.sort(want_logits[first_diff - 1].astype(np.float64))
        margin = l[-1] - l[-2]
    assert first_diff is None or first_diff > n_prompt + 32, f"token mismatch at {first_diff}, top-1/top-2 margin {margin}"
    upto = steps if first_diff is None else first_diff
    worst = max(rel_l2(got_logits[p], want_logits[p]) for p in range(upto))
    assert worst <= 1e-2, worst


# Shapes that send the fused schedule's QKV launch (RMSNorm and rotation inside; reachable through the model only) down
# its different forms: rows of 2.5 and 1.25 passes of 64 lanes (two and four rows side by side in a wave), of less than
# one pass, grouped queries with each of those, and the three head sizes.
SHAPES_FUSED = {
    "rows-of-2560": dict(dim=2560, hidden_dim=3456, n_layers=1, n_heads=20, n_kv_heads=20),
    "rows-of-2560-grouped": dict(dim=2560, hidden_dim=3456, n_layers=2, n_heads=20, n_kv_heads=4),
    "rows-of-640": dict(dim=640, hidden_dim=1728, n_layers=2, n_heads=5, n_kv_heads=5),
    "rows-of-640-grouped": dict(dim=640, hidden_dim=1728, n_layers=2, n_heads=5, n_kv_heads=1),
    "rows-of-1280": dict(dim=1280, hidden_dim=3456, n_layers=1, n_heads=10, n_kv_heads=2),
    "heads-of-64": dict(dim=320, hidden_dim=864, n_layers=2, n_heads=5, n_kv_heads=5),
    "heads-of-256": dict(dim=768, hidden_dim=2048, n_layers=2, n_heads=3, n_kv_heads=1),
}


@pytest.mark.parametrize("shape", sorted(SHAPES_FUSED))
def test_model_shapes_through_the_fused_schedule(ctx, shape):
    cfg = dict(SHAPES_FUSED[shape], vocab_size=512, seq_len=40, rope_theta=10000.0)
    img = synth.make_model_image(cfg, seed=11, scale_mult=0.5)
    t = A.Transformer(ctx, image=img)
    o = oracle.Model(img)
    try:
        prompt = synth.prompt_tokens(4, 5, cfg["vocab_size"])
        kv_dim = cfg["dim"] * cfg["n_kv_heads"] // cfg["n_heads"]
        for mode, graph in ((A.SCHEDULE_FUSED, False), (A.SCHEDULE_FUSED, True), (A.SCHEDULE_REFERENCE, False)):
            t.reset(prompt)
            o.reset(prompt)
            for step in range(12):
                t.ctx.sync()
                gen = step >= len(prompt) - 1
                t.forward(gen_token=gen, use_graph=graph, mode=mode)
                o.forward(gen_token=gen)
                t.ctx.sync()
                got, want = f16(t.download("logits", cfg["vocab_size"])), f16(o.buffer("logits", cfg["vocab_size"]))
                assert rel_l2(got, want) <= 1e-2, (shape, mode, graph, step)
                if t.token(step + 1) != o.tokens(step + 2)[step + 1]:  # a flip on a near tie: follow the oracle
                    top = np.sort(want.astype(np.float64))
                    assert top[-1] - top[-2] <= 4 * np.abs(got.astype(np.float64) - want.astype(np.float64)).max(), (shape, step)
                    t.set_pos(step + 1, o.tokens(step + 2)[step + 1])
            n = 12 * kv_dim
            for name in ("key_cache", "value_cache"):
                assert rel_l2(f16(t.download(name, n)), f16(o.buffer(name, n))) <= 1e-2, (shape, mode, name)
            assert rel_l2(f16(t.download("q", cfg["dim"])), f16(o.buffer("q", cfg["dim"]))) <= 1e-2
    finally:
        t.close()
        o.close()


def test_capture_ahead_of_time_changes_nothing(ctx):
    """Recording every bin up front (seq_len 300: bins 128, 256 and the model's own length) leaves the run state alone
    and gives the tokens of a run that records on first visit; the bins are crossed inside the run."""
    cfg = dict(dim=256, hidden_dim=768, n_layers=2, n_heads=2, n_kv_heads=2, vocab_size=512, seq_len=300, rope_theta=10000.0)
    img = synth.make_model_image(cfg, seed=8, scale_mult=0.25)
    prompt = synth.prompt_tokens(8, 4, cfg["vocab_size"])
    o = oracle.Model(img)
    want, _, _ = o.generate(prompt, 299, ignore_eos=True)
    o.close()
    runs = []
    for ahead in (False, True):
        t = A.Transformer(ctx, image=img)
        t.reset(prompt)
        if ahead:
            t.forward(False, True, A.SCHEDULE_FUSED)  # something in flight and a position other than 0
            t.capture(cfg["seq_len"], A.SCHEDULE_FUSED)
            t.capture(cfg["seq_len"], A.SCHEDULE_REFERENCE)
            ctx.sync()
            assert t.pos == 1
            t.reset(prompt)
        toks, pos = t.generate(prompt, 299, ignore_eos=True, use_graph=True, mode=A.SCHEDULE_FUSED)
        assert pos == 299
        runs.append(toks)
        with pytest.raises(A.AwqError):
            t.capture(cfg["seq_len"] + 1)
        t.close()
    assert runs[0] == runs[1]
    agree = next((i for i in range(300) if runs[0][i] != want[i]), 300)
    assert agree > 4 + 32, agree  # greedy tokens as the oracle's well past the benchmark's 32 steps


def test_context_and_model_handed_between_host_threads():
    """The reference allocates on one short-lived thread, issues every launch from another and tears down from the
    main thread (llama2_q4.cu:613-623, 685, 776-783).  Same hand-off through the C-ABI: context + model created on
    thread A (which exits), decode loop on thread B under graph replay and eagerly, prefill on thread C, free on
    thread D; the tokens are the oracle's."""
    import threading

    cfg = dict(SMALL, hidden_dim=2816)  # multiples of 128, as the batched prefill needs
    img = synth.make_model_image(cfg, seed=11, scale_mult=0.25)
    prompt = synth.prompt_tokens(11, 6, cfg["vocab_size"])
    o = oracle.Model(img)
    want, _, _ = o.generate(prompt, 40, ignore_eos=True)
    o.close()
    box, errors = {}, []

    def on_thread(fn):
        def run():
            try:
                fn()
            except BaseException as e:  # surfaced in the main thread below
                errors.append(e)

        th = threading.Thread(target=run)
        th.start()
        th.join()
        assert not errors, errors

    def create():
        box["ctx"] = A.Context(0)
        box["t"] = A.Transformer(box["ctx"], image=img)

    def decode(graph):
        def fn():
            box[graph] = box["t"].generate(prompt, 40, ignore_eos=True, use_graph=graph, mode=A.SCHEDULE_FUSED)[0]

        return fn

    def prefill():
        t = box["t"]
        t.reset(prompt)
        t.prefill(len(prompt), gen_token=True)
        box["ctx"].sync()
        box["next"] = t.token(len(prompt))

    def destroy():
        box["t"].close()
        box["ctx"].close()

    on_thread(create)
    on_thread(decode(True))
    on_thread(decode(False))
    on_thread(prefill)
    on_thread(destroy)
    agree = next((i for i in range(41) if box[True][i] != want[i]), 41)
    assert agree > 6 + 32, agree
    assert box[True] == box[False]
    assert box["next"] == want[len(prompt)]


def test_eos_stops_generation(pair):
    """The loop breaks when token 2 is read back (llama2_q4.cu:730)."""
    cfg, t, o = pair
    prompt = [5, 2, 9]  # EOS inside the prompt: both stop when it is read back at pos 1
    got_tokens, got_pos = t.generate(prompt, 10)
    want_tokens, want_pos, _ = o.generate(prompt, 10)
    assert got_pos == want_pos == 1


def test_load_errors(ctx):
    img = synth.make_model_image(TINY, seed=0)
    with pytest.raises(A.AwqError):
        A.Transformer(ctx, image=img[:1000])  # short image: "error reading weights"
    bad = img.copy()
    bad[:4] = np.array([-5], dtype=np.int32).view(np.uint8)
    with pytest.raises(A.AwqError):
        A.Transformer(ctx, image=bad)
    with pytest.raises(A.AwqError):
        A.Transformer(ctx, path="/nonexistent/model.bin")


def test_load_file_equals_image(ctx, tmp_path):
    img = synth.make_model_image(TINY, seed=3)
    p = tmp_path / "m.bin"
    img.tofile(p)
    a = A.Transformer(ctx, image=img)
    b = A.Transformer(ctx, path=str(p))
    prompt = synth.prompt_tokens(4, 4, TINY["vocab_size"])
    ta, _ = a.generate(prompt, 20, ignore_eos=True)
    tb, _ = b.generate(prompt, 20, ignore_eos=True)
    assert ta == tb
    a.close()
    b.close()


def test_persistent_schedule_rejects_unsupported_shape(ctx):
    """hidden_dim 1376 has an odd number of groups per row: the persistent kernel declines, the others run."""
    cfg = dict(dim=512, hidden_dim=1376, n_layers=1, n_heads=4, n_kv_heads=4, vocab_size=512, seq_len=32, rope_theta=10000.0)
    t = A.Transformer(ctx, image=synth.make_model_image(cfg, seed=5))
    t.reset([5, 6])
    with pytest.raises(A.AwqError) as e:
        t.forward(False, False, A.SCHEDULE_PERSISTENT)
    assert e.value.code == -2
    t.forward(False, False, A.SCHEDULE_FUSED)
    t.ctx.sync()
    assert t.pos == 1
    t.close()


def test_schedules_can_be_mixed_within_a_sequence(pair):
    """Tokens and positions stay consistent when consecutive tokens use different schedules."""
    cfg, t, o = pair
    prompt = synth.prompt_tokens(7, 4, cfg["vocab_size"])
    want, _, _ = o.generate(prompt, 24, ignore_eos=True)
    t.reset(prompt)
    modes = [A.SCHEDULE_PERSISTENT, A.SCHEDULE_FUSED, A.SCHEDULE_REFERENCE]
    for pos in range(24):
        t.ctx.sync()
        t.forward(pos >= len(prompt) - 1, False, modes[pos % 3])
    t.ctx.sync()
    got = [t.token(i) for i in range(25)]
    assert got == want


def test_fused_gate_up_with_more_row_groups_than_workgroups(ctx):
    """hidden_dim 4480 gives 1120 row groups of 4: more than the 3 workgroups per compute unit that the norm-fused
    gate/up kernel launches, so its workgroups walk 1 or 2 groups each on a 256-CU part (and the last group is the ragged one)."""
    cfg = dict(dim=256, hidden_dim=4480, n_layers=1, n_heads=2, n_kv_heads=2, vocab_size=512, seq_len=48, rope_theta=10000.0)
    img = synth.make_model_image(cfg, seed=5)
    t = A.Transformer(ctx, image=img)
    o = oracle.Model(img)
    try:
        prompt = synth.prompt_tokens(3, 4, cfg["vocab_size"])
        t.reset(prompt)
        o.reset(prompt)
        for _ in range(2):
            t.forward(gen_token=False, use_graph=False, mode=A.SCHEDULE_FUSED)
            o.forward(gen_token=False)
        t.ctx.sync()
        got, want = f16(t.download("hb", cfg["hidden_dim"])), f16(o.buffer("hb", cfg["hidden_dim"]))
        assert rel_l2(got, want) <= 1e-3
        want_tokens, _, _ = o.generate(prompt, 24, ignore_eos=True)
        got_tokens, _ = t.generate(prompt, 24, ignore_eos=True, use_graph=False, mode=A.SCHEDULE_FUSED)
        assert got_tokens == want_tokens
    finally:
        t.close()
        o.close()


# heads, head size, key heads, positions: launch sizes past 256.  Up to 1024 (heads of 64) and 512 (of 128) positions are one request
# of a head; past them, and for heads of 256 at once, they are split over two to four workgroups: the first such sizes, ranges that
# fill no or several rounds of requests (512, 256 and 128 positions for heads of 64, 128 and 256), last ranges that are short, two
# ranges a head (128 heads), 13 waves in the O projection (52 heads); few heads of 128 and 256 past 1279, where P.V is a launch of its own
@pytest.mark.parametrize(
    "heads,head,kv,positions",
    [(4, 64, 2, (128, 256, 300, 1022, 1023, 1024, 1025, 1100, 1535, 1536, 2047, 4500)),
     (4, 128, 4, (129, 255, 256, 511, 512, 513, 767, 768, 1023, 1024, 3000, 5000)),
     (8, 128, 1, (256, 257, 512, 700)), (2, 256, 1, (256, 512, 1500, 2600)), (128, 64, 128, (257, 1100)),
     (32, 128, 8, (1025, 2047, 4500)), (32, 256, 8, (1500, 2600)), (52, 128, 52, (300, 600, 1100))],
)
def test_attention_of_long_contexts_in_one_launch(ctx, heads, head, kv, positions):
    """The fused schedule's attention in ranges, put together by the O projection, against the reference schedule's separate
    launches on the same cache.  fp16 activations behind it differ by single roundings (under 1e-3 in the norm); values that
    grow with the position make a range that is missed or weighted wrongly a difference of several per cent."""
    dim, seq = heads * head, 5120
    cfg = dict(dim=dim, hidden_dim=256, n_layers=1, n_heads=heads, n_kv_heads=kv, vocab_size=512, seq_len=seq, rope_theta=10000.0)
    t = A.Transformer(ctx, image=synth.make_model_image(cfg, seed=5))
    rng = np.random.default_rng(heads * head + kv)
    t.buffer("key_cache", seq * kv * head * 2).write(rng.standard_normal((seq, kv * head)).astype(np.float16))
    rows = rng.standard_normal((seq, kv * head)) + 8 * np.arange(seq)[:, None] / seq - 2
    t.buffer("value_cache", seq * kv * head * 2).write(rows.astype(np.float16))
    for pos in positions:
        logits, scores = {}, {}
        for mode, graph in ((A.SCHEDULE_REFERENCE, False), (A.SCHEDULE_FUSED, False), (A.SCHEDULE_FUSED, True)):
            t.set_pos(pos, 7)
            t.forward_logits(use_graph=graph, mode=mode)
            ctx.sync()
            logits[mode, graph] = t.download("logits", cfg["vocab_size"]).view(np.float16).astype(np.float64)
            scores[mode, graph] = t.download("att", heads * (pos + 1)).view(np.float16)
        want = logits[A.SCHEDULE_REFERENCE, False]
        assert np.isfinite(want).all()
        for key in ((A.SCHEDULE_FUSED, False), (A.SCHEDULE_FUSED, True)):
            assert rel_l2(logits[key], want) <= 4e-3, (pos, key)
            assert rel_l2(scores[key], scores[A.SCHEDULE_REFERENCE, False]) <= 2e-3, (pos, key)
    t.close()


# sizes of the launch past 256 positions: ranges for heads of 256, for heads of 64 one request up to 1024; that is also where the reference's
# maximum starts elsewhere
@pytest.mark.parametrize("heads,head,kv", [(8, 64, 2), (2, 256, 1)], ids=["heads-of-64", "heads-of-256"])
@pytest.mark.parametrize("size", [257, 301, 501, 1022, 1023, 1024, 1025, 1279])
def test_decode_scores_far_below_zero(ctx, heads, head, kv, size):
    """A constant added to every score changes no softmax: scores of -4 .. 4 and the same ones 20, 95 and 150 lower, whose
    exponentials are small, denormal and zero in fp32.  All are multiples of an eighth, which fp16 and its key rows hold, and the
    pair of dimensions in use turns by 1.5e-3 over the context, which moves a score by 1e-4 at most.  What may differ is five
    roundings to fp16 on the way to the second layer's row (6e-4 together): 1e-3."""
    cfg = dict(dim=heads * head, hidden_dim=256, n_layers=2, n_heads=heads, n_kv_heads=kv, vocab_size=512, seq_len=1280, rope_theta=1e6)
    rng = np.random.default_rng(size)
    prompt = [_token(PROFILES["by-slice"](i, size), rng, cfg["vocab_size"]) for i in range(size)]
    outs = []
    for offset in (0.0, -20.0, -95.0, -150.0):
        t = A.Transformer(ctx, image=_designed(cfg, 66, 4.0, offset))
        t.reset(prompt)
        t.prefill(size - 1, gen_token=False)
        t.forward(True, use_graph=True)
        ctx.sync()
        outs.append([rows[1, size - 1] for rows in _rows(t, cfg, size)] + [f16(t.download("logits", cfg["vocab_size"]))])
        t.close()
    for got in outs[1:]:
        for a, b in zip(got, outs[0]):
            assert np.isfinite(a).all() and rel_l2(a, b) <= 1e-3


@pytest.mark.parametrize("heads,head,kv,pos", [(4, 64, 2, 300), (4, 64, 2, 1100), (8, 128, 2, 700), (2, 256, 1, 900), (32, 128, 8, 2100), (4, 128, 4, 2100)])
def test_rows_past_the_position_do_not_enter(ctx, heads, head, kv, pos):
    """Loads past a range's end repeat its last row, and what lies behind the position (an earlier, longer conversation) is not
    read: NaN there changes no bit.  NaN and infinities of the rows that count reach the logits, as in the reference schedule."""
    seq, row = 2304, kv * head
    cfg = dict(dim=heads * head, hidden_dim=256, n_layers=1, n_heads=heads, n_kv_heads=kv, vocab_size=512, seq_len=seq, rope_theta=10000.0)
    t = A.Transformer(ctx, image=synth.make_model_image(cfg, seed=6))
    rng = np.random.default_rng(pos)
    rows = {name: rng.standard_normal((seq, row)).astype(np.float16) for name in ("key_cache", "value_cache")}

    def logits(mode, graph, **changes):
        for name, r in rows.items():
            r = r.copy()
            for at, value in changes.get(name, ()):
                r[at] = value
            t.buffer(name, seq * row * 2).write(r)
        t.set_pos(pos, 7)
        t.forward_logits(use_graph=graph, mode=mode)
        ctx.sync()
        return f16(t.download("logits", cfg["vocab_size"])).copy()

    behind = slice(pos + 1, None)
    for graph in (False, True):
        want = logits(A.SCHEDULE_FUSED, graph)
        assert np.isfinite(want).all()
        for value in (np.nan, np.inf):
            got = logits(A.SCHEDULE_FUSED, graph, key_cache=[(behind, value)], value_cache=[(behind, value)])
            assert np.array_equal(got.view(np.uint16), want.view(np.uint16))
    # a key that is NaN, and a value that is infinite, in the first range and in the last
    for at in (3, pos - 1):
        for change in (dict(key_cache=[((at, row - 1), np.nan)]), dict(value_cache=[((at, row - 1), np.inf)])):
            for mode in (A.SCHEDULE_REFERENCE, A.SCHEDULE_FUSED):
                assert not np.isfinite(logits(mode, False, **change)).any(), (at, change, mode)
    t.close()
