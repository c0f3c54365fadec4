"""Gemodra through the engine against the plain implementation (``plain_gemodra.py``,
float64, whole sequences, one function per mechanism, keys and values of every head formed
from the latent vectors).

float32 runs are held to the plain logits row by row (root mean square of the difference
over the vocabulary, means taken off, relative to the logits' own spread); every schedule,
cut and batch is held to the same bound.  A bfloat16 run chooses experts from a rounded
input: where two choice scores are closer than that rounding a token goes to another expert
than in float64, and the test weights are drawn with routers far from flat on purpose, so
single rows may differ visibly (measured: one row in some hundreds, by as much as the
logits' own spread).  bfloat16 rows are therefore held to the plain logits by their median
and their ninth decile, and only a few in a hundred may be far off; and how a bfloat16
request was cut and batched must not show beyond rounding: every schedule is held to the
whole prompts' run in the same way."""

import copy
import math

import pytest
import torch

import engine_util as eu
import gemodra_util as gu
import plain_gemodra as plain

pytestmark = pytest.mark.gpu

F32_BOUND = 1e-4
BF16_MEDIAN, BF16_DECILE = 0.04, 0.12
BF16_FAR, BF16_FAR_SHARE = 0.3, 0.03          # rows further off than this, and how many may be
BF16_BETWEEN_MEDIAN, BF16_BETWEEN_DECILE = 0.02, 0.06


def build(cfg, seed=0, dtype="float32", tensors=None):
    from zig_ai_amd.engine import DecoderModel
    d, tensors = gu.folder(cfg, seed, tensors)
    return DecoderModel.from_folder(d, dtype), tensors


def runner_for(model, page_size=4, tokens=256, slots=4, graphs=True):
    from zig_ai_amd.engine import ModelRunner
    return ModelRunner(model, page_size=page_size, num_pages=max(1, -(-tokens // page_size)),
                       num_slots=slots, use_graphs=graphs)


def plain_logits(cfg, tensors, prompts):
    return [plain.forward(cfg, tensors, p).float() for p in prompts]


def worst(got, want):
    return float(gu.row_error(got, want).max())


def assert_bfloat16_close(got, want, what=None):
    e = gu.row_error(got, want)
    found = (float(e.median()), float(e.quantile(0.9)), float((e > BF16_FAR).double().mean()))
    assert found[0] < BF16_MEDIAN and found[1] < BF16_DECILE and found[2] <= BF16_FAR_SHARE, \
        (what, found)


def assert_bfloat16_same_run(got, base, what=None):
    e = gu.row_error(got, base)
    found = (float(e.median()), float(e.quantile(0.9)))
    assert found[0] < BF16_BETWEEN_MEDIAN and found[1] < BF16_BETWEEN_DECILE, (what, found)


# ----------------------------------------------------------- each mechanism alone
SMALL = gu.plain_latent(heads=2, dim=8, vdim=8, kv_rank=16, q_rank=8)
ALONE = {
    "rotated": gu.one_layer("latent_attention", gu.latent(), side=0, softcap=0.0),
    "rotated, a part of the part turned": gu.one_layer(
        "latent_attention", gu.latent(heads=2, dim=24, vdim=8, kv_rank=40, q_rank=16, rot_dim=16,
                                      rot_dims=6, base=40.0), side=0, softcap=0.0),
    "rotated, one head, two rotated elements": gu.one_layer(
        "latent_attention", gu.latent(heads=1, dim=40, vdim=48, kv_rank=24, q_rank=8, rot_dim=2),
        side=0, softcap=0.0),
    "rotated, many heads": gu.one_layer(
        "latent_attention", gu.latent(heads=40, dim=8, vdim=8, kv_rank=72, q_rank=16, rot_dim=8),
        side=0, softcap=0.0, width=64),
    "unrotated": gu.one_layer("latent_attention_2", gu.plain_latent(), side=0, softcap=0.0),
    "unrotated, one head": gu.one_layer("latent_attention_2", gu.plain_latent(
        heads=1, dim=16, vdim=40, kv_rank=8, q_rank=32), side=0, softcap=0.0),
    "unrotated, a wide latent": gu.one_layer("latent_attention_2", gu.plain_latent(
        heads=3, dim=16, vdim=16, kv_rank=320, q_rank=16), side=0, softcap=0.0, width=64),
    "experts in groups": gu.one_layer("latent_attention_2", SMALL, gu.moe(
        ff=16, experts=9, identity=3, top=3, groups=(4, 2), shared=0), side=0, softcap=0.0),
    "experts, no groups, a shared one": gu.one_layer("latent_attention_2", SMALL, gu.moe(
        ff=24, experts=5, identity=0, top=2, shared=40), side=0, softcap=0.0),
    "all outputs chosen": gu.one_layer("latent_attention_2", SMALL, gu.moe(
        ff=8, experts=2, identity=1, top=3, shared=0, scale=0.7), side=0, softcap=0.0),
    "identity outputs only": gu.one_layer("latent_attention_2", SMALL, gu.moe(
        experts=0, identity=4, top=2, groups=(2, 1), shared=8), side=0, softcap=0.0),
    "one group kept": gu.one_layer("latent_attention_2", SMALL, gu.moe(
        ff=16, experts=6, identity=2, top=2, groups=(4, 1), shared=0), side=0, softcap=0.0),
    "token input": gu.one_layer("latent_attention_2", SMALL, None, side=12, softcap=0.0),
    "capped logits": gu.one_layer("latent_attention_2", SMALL, None, side=0, softcap=1.5),
}


@pytest.mark.parametrize("name", sorted(ALONE))
def test_mechanism_alone(name):
    cfg = ALONE[name]
    model, tensors = build(cfg, seed=3)
    prompts = [gu.tokens(70, cfg["vocab"], 1), gu.tokens(5, cfg["vocab"], 2)]
    want = plain_logits(cfg, tensors, prompts)
    runner = runner_for(model)
    got = eu.run_schedule(runner, prompts, eu.whole([len(p) for p in prompts]))
    for g, w in zip(got, want):
        assert worst(g, w) < F32_BOUND
    # the same, token by token from the first token on: the cache alone
    got = eu.run_schedule(runner, prompts, eu.bulk_then_single([len(p) for p in prompts], tail=10 ** 6))
    for g, w in zip(got, want):
        assert worst(g, w) < F32_BOUND


def test_every_mechanism_counts():
    """The plain implementation without one mechanism is far from the one with it: the
    weights make each of them visible, so the comparisons above can fail."""
    cfg = gu.TINY_ALL
    tensors = gu.make_tensors(cfg, seed=3)
    prompt = gu.tokens(40, cfg["vocab"], 1)
    want = plain.forward(cfg, tensors, prompt).float()

    def changed(edit_cfg=None, edit_tensors=None):
        c, t = copy.deepcopy(cfg), dict(tensors)
        if edit_cfg:
            edit_cfg(c)
        if edit_tensors:
            edit_tensors(t)
        return worst(plain.forward(c, t, prompt).float(), want)

    def no_sink(t):
        for i in range(4):
            t[f"l{i}.mix.sink"] = torch.full_like(t[f"l{i}.mix.sink"], -60.0)

    def no_correction(t):
        for i in (0, 1, 3):
            t[f"l{i}.mlp.correction"] = torch.zeros_like(t[f"l{i}.mlp.correction"])

    def no_groups(c):
        for i in (0, 3):
            del c["layers"][i]["mlp"]["router"]["groups"]

    def no_side(c):
        del c["token_side"]

    def no_cap(c):
        del c["logit_softcap"]

    def other_base(c):
        c["layers"][0]["mixer"]["rot"]["base"] = 3000.0

    def no_shared_gate(t):
        t["l0.mlp.shared.sg"] = torch.zeros_like(t["l0.mlp.shared.sg"])

    def no_embed_norm(t):
        t["embed.norm"] = torch.ones_like(t["embed.norm"])

    for name, kw in (("sink", {"edit_tensors": no_sink}), ("correction", {"edit_tensors": no_correction}),
                     ("groups", {"edit_cfg": no_groups}), ("token input", {"edit_cfg": no_side}),
                     ("cap", {"edit_cfg": no_cap}), ("base", {"edit_cfg": other_base}),
                     ("shared gate", {"edit_tensors": no_shared_gate}),
                     ("embedding norm", {"edit_tensors": no_embed_norm})):
        assert changed(**kw) > 0.02, name


# ------------------------------- sizes that are multiples of nothing the kernels like
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_awkward_sizes(dtype):
    cfg = gu.config([
        gu.layer("latent_attention", gu.latent(heads=3, dim=12, vdim=20, kv_rank=28, q_rank=12,
                                               rot_dim=6, base=77.0),
                 gu.moe(ff=20, experts=7, identity=2, top=3, groups=(3, 2), shared=12)),
        gu.layer("latent_attention_2", gu.plain_latent(heads=7, dim=10, vdim=6, kv_rank=18, q_rank=14),
                 gu.moe(ff=12, experts=2, identity=0, top=1, shared=0)),
        gu.layer("latent_attention", gu.latent(heads=70, dim=8, vdim=8, kv_rank=16, q_rank=24,
                                               rot_dim=8), None),
    ], width=36, vocab=53, side=6, softcap=9.0, mult=0.7)
    model, tensors = build(cfg, seed=17, dtype=dtype)
    lengths = [50, 3, 21]
    prompts = [gu.tokens(n, cfg["vocab"], 30 + i) for i, n in enumerate(lengths)]
    want = plain_logits(cfg, tensors, prompts)
    base = None
    for name, schedule in (("whole", eu.whole(lengths)),
                           ("portions", eu.changing_portions(lengths, seed=2)),
                           ("mixed", eu.mixed(lengths, seed=3, max_live=3, decode_tail=8))):
        got = eu.run_schedule(runner_for(model, page_size=8, tokens=128, slots=3), prompts, schedule)
        if dtype == "float32":
            for g, w in zip(got, want):
                assert worst(g, w) < F32_BOUND, name
        else:
            assert_bfloat16_close(torch.cat(got), torch.cat(want), name)
            base = base or got
            assert_bfloat16_same_run(torch.cat(got), torch.cat(base), name)


# -------------------------------------------------------- schedules of whole models
LENGTHS = [150, 37, 9, 1, 75, 130, 2]


def schedules(lengths):
    return {
        "whole": eu.whole(lengths),
        "bulk + tail": eu.bulk_then_single(lengths, tail=40),
        "portions": eu.changing_portions(lengths, seed=1),
        "portions of two": eu.changing_portions(lengths, seed=0, sizes=(2, 2, 3, 2, 17)),
        "mixed": eu.mixed(lengths, seed=2, max_live=4, decode_tail=20),
        "mixed, three live": eu.mixed(lengths, seed=5, max_live=3, decode_tail=45),
    }


@pytest.mark.parametrize("which", ["all", "other"])
@pytest.mark.parametrize("page_size", [4, 16])
def test_schedules_float32(which, page_size):
    cfg = gu.TINY_ALL if which == "all" else gu.TINY_OTHER
    model, tensors = build(cfg, seed=11)
    prompts = [gu.tokens(n, cfg["vocab"], 20 + i) for i, n in enumerate(LENGTHS)]
    want = plain_logits(cfg, tensors, prompts)
    for name, schedule in schedules(LENGTHS).items():
        # a pool for the most tokens live at any time: pages are used again
        peak = eu.peak_tokens(LENGTHS, schedule, round_to=max(16, page_size))
        runner = runner_for(model, page_size=page_size, tokens=peak, slots=4)
        got = eu.run_schedule(runner, prompts, schedule)
        for i, (g, w) in enumerate(zip(got, want)):
            assert worst(g, w) < F32_BOUND, (name, i)
        if "mixed" in name:
            assert runner.cache.pages_reused > 0
        assert len(runner.cache.requests) == 0


@pytest.mark.parametrize("which", ["all", "other"])
def test_schedules_bfloat16(which):
    cfg = gu.TINY_ALL if which == "all" else gu.TINY_OTHER
    model, tensors = build(cfg, seed=11, dtype="bfloat16")
    prompts = [gu.tokens(n, cfg["vocab"], 20 + i) for i, n in enumerate(LENGTHS)]
    want = plain_logits(cfg, tensors, prompts)
    base = None
    for name, schedule in schedules(LENGTHS).items():
        peak = eu.peak_tokens(LENGTHS, schedule, round_to=16)
        runner = runner_for(model, page_size=16, tokens=peak, slots=4)
        got = eu.run_schedule(runner, prompts, schedule)
        assert_bfloat16_close(torch.cat(got), torch.cat(want), name)
        if base is None:
            base = got
        assert_bfloat16_same_run(torch.cat(got), torch.cat(base), name)


# ------------------------------------------------ configurations drawn at random
@pytest.mark.parametrize("seed", range(10))
def test_random_configurations(seed):
    cfg = gu.random_config(seed)
    lengths = [70, 1, 33, 12, 2]
    prompts = [gu.tokens(n, cfg["vocab"], 90 + i) for i, n in enumerate(lengths)]
    model, tensors = build(cfg, seed=seed)
    want = plain_logits(cfg, tensors, prompts)
    for name, schedule in (("whole", eu.whole(lengths)),
                           ("portions", eu.changing_portions(lengths, seed=seed)),
                           ("mixed", eu.mixed(lengths, seed=seed, max_live=3, decode_tail=9))):
        peak = eu.peak_tokens(lengths, schedule, round_to=16)
        runner = runner_for(model, page_size=4 if seed % 2 else 16, tokens=peak, slots=3)
        got = eu.run_schedule(runner, prompts, schedule)
        for i, (g, w) in enumerate(zip(got, want)):
            assert worst(g, w) < 3 * F32_BOUND, (name, i, cfg)
    # the same model in bfloat16 runs (odd widths fall back to 32-bit weights) and agrees
    # with itself across schedules
    model16, _ = build(cfg, seed=seed, dtype="bfloat16")
    base = None
    for schedule in (eu.whole(lengths), eu.mixed(lengths, seed=seed, max_live=3, decode_tail=9)):
        got = eu.run_schedule(runner_for(model16, page_size=16, tokens=256, slots=3), prompts, schedule)
        assert all(torch.isfinite(g).all() for g in got)
        base = base or got
        assert_bfloat16_same_run(torch.cat(got), torch.cat(base), cfg)


# --------------------------------- the causal edge, with scores that stand out
def sharp_cfg(kind):
    # a scale that makes the softmax all but choose one key: a key wrongly seen or wrongly
    # hidden then takes or loses nearly all of a query's weight
    mixer = gu.latent(heads=2, dim=16, vdim=16, kv_rank=24, q_rank=16, rot_dim=8, base=100.0,
                      scale=3.0) if kind == "latent_attention" else \
        gu.plain_latent(heads=2, dim=16, vdim=16, kv_rank=24, q_rank=16, scale=3.0)
    return gu.one_layer(kind, mixer, None, side=0, softcap=0.0)


def plain_with_reach(cfg, tensors, prompt, reach):
    """The plain model with every query seeing one key fewer (-1: not itself) or one more
    (+1: its successor too) than it should."""
    real = plain.latent_attention
    plain.latent_attention = lambda *a, **k: real(*a, reach=reach, **k)
    try:
        return plain.forward(cfg, tensors, prompt).float()
    finally:
        plain.latent_attention = real


@pytest.mark.parametrize("kind", ["latent_attention", "latent_attention_2"])
def test_causal_edge(kind):
    cfg = sharp_cfg(kind)
    model, tensors = build(cfg, seed=5)
    n = 90
    prompts = [gu.tokens(n, cfg["vocab"], 7)]
    want = plain_logits(cfg, tensors, prompts)[0]
    # the test can see an edge that is one token off
    for reach in (-1, 1):
        assert worst(plain_with_reach(cfg, tensors, prompts[0], reach), want) > 0.05
    for page_size in (4, 16):
        for name, schedule in (("whole", eu.whole([n])),
                               ("decoded", eu.bulk_then_single([n], tail=n - 3)),
                               ("portions", eu.changing_portions([n], sizes=(5, 2, 16, 3, 17, 15, 1)))):
            runner = runner_for(model, page_size=page_size, tokens=128)
            got = eu.run_schedule(runner, prompts, schedule)[0]
            assert worst(got, want) < 1e-3, (name, page_size)


# ----------------------------------------------------------------- far tokens count
def far_prompt(cfg, tensors, n, place):
    """A prompt of ``n`` tokens and the same with another token at ``place``, made so that the
    last rows of the plain logits differ clearly: the body repeats three ids, the token at
    ``place`` occurs nowhere else, and the last eight tokens are one id whose queries it
    draws (both found by trying the ids kept aside for this)."""
    V = cfg["vocab"]
    body = [t % 3 for t in gu.tokens(n, V, 3)]
    best = None
    for tail in range(V - 16, V - 8):
        for cand in range(V - 8, V):
            a = list(body)
            a[-8:] = [tail] * 8
            b = list(a)
            a[place] = cand
            wa, wb = plain.forward(cfg, tensors, a).float(), plain.forward(cfg, tensors, b).float()
            d = worst(wb[-8:], wa[-8:])
            if best is None or d > best[0]:
                best = (d, a, b, wa, wb)
            if d > 0.1:
                return best
    return best


@pytest.mark.parametrize("kind", ["latent_attention", "latent_attention_2"])
def test_far_tokens_reach_the_end(kind):
    cfg = sharp_cfg(kind)
    tensors = gu.make_tensors(cfg, seed=9)
    tensors["l0.mix.sink"] = torch.full_like(tensors["l0.mix.sink"], -4.0)
    model, tensors = build(cfg, tensors=tensors)
    n = 600
    d, a, b, wa, wb = far_prompt(cfg, tensors, n, place=1)
    assert d > 0.02           # the second token still shows at the end, among hundreds
    for prompt, want in ((a, wa), (b, wb)):
        for page_size, schedule in ((16, eu.whole([n])), (4, eu.bulk_then_single([n], tail=40)),
                                    (16, eu.changing_portions([n], sizes=(33, 2, 64, 17, 200)))):
            got = eu.run_schedule(runner_for(model, page_size=page_size, tokens=640), [prompt],
                                  schedule)[0]
            assert worst(got, want) < F32_BOUND
    # nothing is left of a request whose pages are taken again: b after a in the same pool
    runner = runner_for(model, page_size=16, tokens=640, slots=1)
    for prompt, want in ((a, wa), (b, wb), (a, wa)):
        got = eu.run_schedule(runner, [prompt], eu.bulk_then_single([n], tail=5))[0]
        assert worst(got, want) < F32_BOUND
    assert runner.cache.pages_reused > 0


# --------------------------------------------------------------------- the sink
@pytest.mark.parametrize("kind", ["latent_attention", "latent_attention_2"])
def test_sinks_that_take_most_of_the_weight(kind):
    cfg = sharp_cfg(kind)
    cfg["layers"][0]["mixer"]["scale"] = 0.2
    tensors = gu.make_tensors(cfg, seed=2)
    tensors["l0.mix.sink"] = torch.tensor([3.0, -1.0])
    model, tensors = build(cfg, tensors=tensors)
    lengths = [60, 3]
    prompts = [gu.tokens(n, cfg["vocab"], 4 + i) for i, n in enumerate(lengths)]
    want = plain_logits(cfg, tensors, prompts)
    # a sink that is scaled like a score, or given to the other head, shows
    for other in (torch.tensor([3.0 * 0.2, -0.2]), torch.tensor([-1.0, 3.0])):
        t2 = dict(tensors)
        t2["l0.mix.sink"] = other
        assert worst(plain.forward(cfg, t2, prompts[0]).float(), want[0]) > 0.02
    for schedule in (eu.whole(lengths), eu.bulk_then_single(lengths, tail=30),
                     eu.changing_portions(lengths, sizes=(2, 7, 16))):
        got = eu.run_schedule(runner_for(model), prompts, schedule)
        for g, w in zip(got, want):
            assert worst(g, w) < F32_BOUND


# ------------------------------------------- keys and values formed from the latent rows
# heads of 128, rotated and not, gates of either kind
FORMED = gu.config([
    gu.layer("latent_attention", gu.latent(heads=2, dim=128, vdim=128, kv_rank=64, q_rank=24, rot_dim=64,
                                           rot_dims=32, base=1e4), None),
    gu.layer("latent_attention_2", gu.plain_latent(heads=3, dim=128, vdim=128, kv_rank=40, q_rank=16), None)])


def test_schedules_over_formed_keys(monkeypatch):
    """Whole prompts, portions behind cached tokens, portions beside single tokens and decoding, from pages of 4
    and 16 tokens: the plain logits whichever form a step takes, and those of the same steps all folded."""
    from zig_ai_amd.parts import latent_attention
    model, tensors = build(FORMED, seed=8, dtype="bfloat16")
    lengths = [150, 37, 70, 2, 1]
    prompts = [gu.tokens(n, FORMED["vocab"], 20 + i) for i, n in enumerate(lengths)]
    want = torch.cat(plain_logits(FORMED, tensors, prompts))
    both = set()
    for name, schedule in dict(schedules(lengths), together=[([(0, 0, 60), (1, 0, 37), (2, 0, 66), (3, 0, 2)], [1, 3]),
                                                             ([(0, 60, 148), (2, 66, 68)], []),
                                                             ([(0, 148, 150), (2, 68, 70)], [0, 2]),
                                                             ([(4, 0, 1)], [4])]).items():
        page_size = 4 if len(name) % 2 else 16
        got = []
        for most in (256 << 20, 0):
            monkeypatch.setattr(latent_attention, "FORMING_BYTES", most)
            forms = eu.FormedKeys(2)
            peak = eu.peak_tokens(lengths, schedule, round_to=16)
            runner = runner_for(model, page_size=page_size, tokens=peak, slots=4, graphs=False)
            got.append(torch.cat(eu.run_schedule(runner, prompts, schedule, forms=forms)))
            assert forms.as_the_rule_says(16 if most else 0), name
            both |= {formed for _, formed in forms.steps if most}
            assert_bfloat16_close(got[-1], want, name)
        assert_bfloat16_same_run(got[0], got[1], name)
    assert both == {False, True}


def test_recorded_portions_take_one_form(monkeypatch):
    """Where portions are recorded, a shape's first step, the recorded one with other contexts behind it, and a step
    of that shape with taps all take the kernels that do not hang on the contexts' lengths; larger steps, which
    are never recorded, form keys and values."""
    from zig_ai_amd.engine import ModelRunner, graphs
    model, tensors = build(FORMED, seed=8, dtype="bfloat16")
    prompts = [gu.tokens(120, FORMED["vocab"], 1), gu.tokens(200, FORMED["vocab"], 2)]
    want = plain_logits(FORMED, tensors, prompts)
    monkeypatch.setattr(graphs, "PORTION_GRAPH_MAX_TOKENS", 64)
    make = lambda on: ModelRunner(model, page_size=16, num_pages=32, num_slots=2, portion_graphs=on)
    recorded, plain_run = make(True), make(False)
    schedule = [([(0, a, a + 40)], [0] if a == 80 else []) for a in (0, 40, 80)] + \
        [([(1, a, a + 100)], [1] if a else []) for a in (0, 100)]
    small = lambda forms: {formed for entries, formed in forms.steps if entries[0][0] == 0}
    large = lambda forms: {formed for entries, formed in forms.steps if entries[0][0] == 1}
    first = None
    for _ in range(3):
        forms = eu.FormedKeys(2)
        got = eu.run_schedule(recorded, prompts, schedule, forms=forms)
        assert small(forms) == {False} and large(forms) == {True}
        assert_bfloat16_close(torch.cat(got), torch.cat(want))
        first = first or got
        # (every sum of the two runs is the same but for the cut of the contexts into ranges)
        assert worst(torch.cat(got), torch.cat(first)) < 0.02
    assert recorded.graphs.portion_captures == 1 and recorded.graphs.portion_replays == 8
    for runner, formed in ((recorded, False), (plain_run, True)):
        forms = eu.FormedKeys(2)
        eu.run_schedule(runner, prompts, schedule[:3], forms=forms, streams={})
        assert small(forms) == {formed}


def test_taps_of_formed_steps(monkeypatch):
    """The queries that a step leaves in its taps are the folded ones, whichever form it takes."""
    from zig_ai_amd.parts import latent_attention
    model, _ = build(FORMED, seed=8, dtype="bfloat16")
    prompts = [gu.tokens(61, FORMED["vocab"], 1)]
    schedule = [([(0, 0, 40)], []), ([(0, 40, 41)], []), ([(0, 41, 61)], [0])]
    left = []
    for most in (256 << 20, 0):
        monkeypatch.setattr(latent_attention, "FORMING_BYTES", most)
        forms, streams = eu.FormedKeys(2), {}
        eu.run_schedule(runner_for(model, page_size=16), prompts, schedule, forms=forms, streams=streams)
        assert [formed for _, formed in forms.steps] == [most > 0, False, most > 0]
        left.append(streams[0])
    for layer, (heads, width) in enumerate(((2, 64 + 64), (3, 40))):
        assert all(run[layer + 1]["q"].shape == (61, heads, width) for run in left)
    # (the first layer's queries hang on nothing that the form changes)
    assert torch.equal(left[0][1]["q"], left[1][1]["q"])


def test_forming_with_rows_to_spare(monkeypatch):
    """Keys and values formed for more rows than there are, whatever memory holds there: the logits of just as many."""
    from zig_ai_amd.parts import latent_attention
    model, tensors = build(FORMED, seed=8, dtype="bfloat16")
    lengths = [190, 33]
    prompts = [gu.tokens(n, FORMED["vocab"], 1 + i) for i, n in enumerate(lengths)]
    want = plain_logits(FORMED, tensors, prompts)
    schedule = [([(0, 0, 64)], []), ([(0, 64, 96), (1, 0, 33)], [1]), ([(0, 96, 129)], []), ([(0, 129, 190)], [0])]
    got = []
    for block in (256, 16, 100):
        monkeypatch.setattr(latent_attention, "FORMING_BLOCK", block)
        for size in (1 << 16, 1 << 14):      # (memory that the next tensors are likely to get)
            torch.full((size,), float("nan"), dtype=torch.bfloat16, device="cuda")
        forms = eu.FormedKeys(2)
        got.append(torch.cat(eu.run_schedule(runner_for(model, page_size=16, tokens=256), prompts, schedule,
                                             forms=forms)))
        assert all(formed for _, formed in forms.steps)
        assert_bfloat16_close(got[-1], torch.cat(want), block)
        assert_bfloat16_same_run(got[-1], got[0], block)


def test_forming_meets_no_row_count_that_warm_up_has_not(monkeypatch):
    """A long prompt in portions behind an engine's warm-up: the GEMM library is asked to form keys and values for no
    number of rows that it has not planned, however long the contexts get."""
    from zig_ai_amd.engine import Engine
    from zig_ai_amd.engine.model import walk_parts
    from zig_ai_amd.kernels import ops
    cfg = gu.config([gu.layer("latent_attention", gu.latent(heads=16, dim=128, vdim=128, kv_rank=128, q_rank=24,
                                                            rot_dim=64, base=1e4), None)])
    model, _ = build(cfg, seed=8, dtype="bfloat16")
    weight_of = [p.w_form for b in model.blocks for part in b.parts.values() for p in walk_parts(part)
                 if hasattr(p, "w_form")]
    assert len(weight_of) == 1
    met, library = set(), ops._library_matmul

    def counted(x, weight, *more, **named):
        if weight is weight_of[0]:
            met.add(x.shape[0])
        return library(x, weight, *more, **named)

    monkeypatch.setattr(ops, "_library_matmul", counted)
    engine = Engine(model, page_size=16, num_pages=256, max_num_seqs=2, max_num_batched_tokens=512)
    planned = set(met)
    assert {256 * k for k in range(1, 9)} | {2560, 3072, 3584, 4096, 5120, 8192} <= planned
    met.clear()
    engine.generate([gu.tokens(3100, cfg["vocab"], 1)], max_new_tokens=2, temperature=0.0, eos_token_id=-1)
    assert len(met) >= 4 and met <= planned, (met, planned)


# -------------------------- a long context: ranges of keys, merged, with the sink once
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_context_in_ranges(dtype):
    from zig_ai_amd.kernels import ops
    cfg = gu.config([gu.layer("latent_attention", gu.latent(heads=2, dim=16, vdim=16, kv_rank=64,
                                                            q_rank=16, rot_dim=16, base=1e4), None),
                     gu.layer("latent_attention_2", gu.plain_latent(), None)], side=8)
    model, tensors = build(cfg, seed=4, dtype=dtype)
    n = 1500
    prompts = [gu.tokens(n, cfg["vocab"], 1), gu.tokens(30, cfg["vocab"], 2)]
    want = plain_logits(cfg, tensors, prompts)
    runner = runner_for(model, page_size=16, tokens=1600, graphs=False)
    wants = [list(range(n - 90, n)), list(range(30))]
    steps = [([(0, 0, n - 80)], [])]
    # the long request decodes beside the short one's portions and single tokens
    steps += [([(0, n - 80 + i, n - 79 + i)] + ([(1, 3 * i, 3 * i + 3)] if i < 10 else []),
               [1] if i == 9 else []) for i in range(80)]
    steps[-1] = (steps[-1][0], [0])
    ops.form_log = []
    try:
        got = eu.run_schedule(runner, prompts, steps, wants=wants)
        cut = [r for r in (ops.form_log or []) if r.get("op") == "attention" and r.get("nsplit", 1) > 1]
    finally:
        ops.form_log = None
    if dtype == "float32":
        assert worst(got[0], want[0][n - 90:]) < F32_BOUND
        assert worst(got[1], want[1]) < F32_BOUND
    else:
        assert_bfloat16_close(torch.cat(got), torch.cat([want[0][n - 90:], want[1]]))


# ------------------------------------------------------------------- long decoding
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding(dtype):
    cfg = gu.TINY_ALL
    model, tensors = build(cfg, seed=21, dtype=dtype)
    n = 330
    prompts = [gu.tokens(n, cfg["vocab"], 5)]
    want = plain_logits(cfg, tensors, prompts)[0]
    runner = runner_for(model, page_size=16, tokens=512)       # decode steps replay from graphs
    got = eu.run_schedule(runner, prompts, eu.bulk_then_single([n], tail=300))[0]
    if dtype == "float32":
        assert worst(got, want) < F32_BOUND
    else:
        assert_bfloat16_close(got, want)


# ------------------------------------------- unequal requests together and alone
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_batch_against_each_alone(dtype):
    cfg = gu.TINY_ALL
    model, tensors = build(cfg, seed=2, dtype=dtype)
    lengths = [64, 3, 41, 17]
    prompts = [gu.tokens(n, cfg["vocab"], 40 + i) for i, n in enumerate(lengths)]
    alone = eu.run_schedule(runner_for(model, tokens=256), prompts, eu.whole(lengths))
    together = [([(i, 0, n) for i, n in enumerate(lengths)], list(range(len(lengths))))]
    got = eu.run_schedule(runner_for(model, tokens=256), prompts, together)
    if dtype == "float32":
        assert worst(torch.cat(got), torch.cat(alone)) < F32_BOUND
    else:
        assert_bfloat16_same_run(torch.cat(got), torch.cat(alone))


# ----------------------------------- sizes at which the products run on the matrix cores
def test_wider_model_bfloat16():
    mixer = gu.latent(heads=8, dim=32, vdim=48, kv_rank=128, q_rank=96, rot_dim=32, base=1e5)
    cfg = gu.config([gu.layer("latent_attention", mixer, gu.moe(ff=64, experts=6, identity=2, top=3,
                                                                groups=(4, 2), shared=128)),
                     gu.layer("latent_attention_2", gu.plain_latent(heads=4, dim=64, vdim=32,
                                                                    kv_rank=256, q_rank=64),
                              gu.moe(ff=128, experts=8, identity=0, top=2, shared=0))],
                    width=256, vocab=300, side=32)
    model, tensors = build(cfg, seed=6, dtype="bfloat16")
    lengths = [200, 70, 3]
    prompts = [gu.tokens(n, cfg["vocab"], 50 + i) for i, n in enumerate(lengths)]
    want = plain_logits(cfg, tensors, prompts)
    base = None
    for name, schedule in (("whole", eu.whole(lengths)),
                           ("bulk + tail", eu.bulk_then_single(lengths, tail=60)),
                           ("portions", eu.changing_portions(lengths, seed=3)),
                           ("mixed", eu.mixed(lengths, seed=1, max_live=3, decode_tail=30))):
        runner = runner_for(model, page_size=16, tokens=512, slots=3)
        got = eu.run_schedule(runner, prompts, schedule)
        assert_bfloat16_close(torch.cat(got), torch.cat(want), name)
        base = base or got
        assert_bfloat16_same_run(torch.cat(got), torch.cat(base), name)


# ------------------------------------------- generation through engine and scheduler
def test_greedy_generation():
    from zig_ai_amd.engine import Engine
    cfg = gu.TINY_ALL
    d, tensors = gu.folder(cfg, seed=8)
    engine = Engine(d, dtype="float32", page_size=4, num_pages=128, max_num_seqs=3,
                    max_num_batched_tokens=48, chunk_size=20, max_model_len=256)
    prompts = [gu.tokens(n, cfg["vocab"], 60 + i) for i, n in enumerate([33, 5, 70, 12, 1])]
    outs = engine.generate(prompts, max_new_tokens=20, temperature=0.0)
    assert all(len(o) == 20 for o in outs)
    for p, o in zip(prompts, outs):
        # every chosen token is the plain implementation's choice for the same history
        logits = plain.forward(cfg, tensors, p + o)
        for j, tok in enumerate(o):
            row = logits[len(p) + j - 1]
            assert float(row.max() - row[tok]) <= 1e-3 * float(row.abs().max()), (j, tok)
    assert len(engine.runner.cache.requests) == 0
    engine.runner.cache.check()


def test_generation_bfloat16_runs_through_graphs():
    from zig_ai_amd.engine import Engine
    cfg = gu.TINY_OTHER
    d, tensors = gu.folder(cfg, seed=8)
    engine = Engine(d, dtype="bfloat16", page_size=16, num_pages=64, max_num_seqs=4,
                    max_model_len=256)
    assert engine.runner.graphs is not None        # every part can be recorded
    prompts = [gu.tokens(n, cfg["vocab"], 80 + i) for i, n in enumerate([40, 7, 19])]
    outs = engine.generate(prompts, max_new_tokens=24, temperature=0.0)
    assert all(len(o) == 24 for o in outs)
    good = total = 0
    for p, o in zip(prompts, outs):
        logits = plain.forward(cfg, tensors, p + o)
        for j, tok in enumerate(o):
            row = logits[len(p) + j - 1]
            spread = float(row.max() - row.min())
            good += float(row.max() - row[tok]) <= 0.1 * spread
            total += 1
    # (a token routed to another expert than in float64 may pick another word; rare)
    assert good >= 0.9 * total, (good, total)


def test_trace_replay_and_command_line(tmp_path):
    import json
    import os
    import subprocess
    import sys
    import numpy as np
    cfg = gu.TINY_ALL
    d, tensors = gu.folder(cfg, seed=8)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    prompt, other = gu.tokens(40, cfg["vocab"], 3), gu.tokens(11, cfg["vocab"], 4)
    want = plain.forward(cfg, tensors, prompt).float()
    want_other = plain.forward(cfg, tensors, other).float()
    # portions of one request beside another's, single tokens, a step in which nothing is asked
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": prompt[:25], "want": [3, 24]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": prompt[25:27], "want": []},
                                     {"id": "b", "tokens": other[:10], "want": []}], "end": []},
             {"step": 2, "entries": [{"id": "b", "tokens": other[10:], "want": [0]},
                                     {"id": "a", "tokens": prompt[27:], "want": [12]}], "end": ["a", "b"]}]
    out = subprocess.run([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", d,
                          "--dtype", "float32", "--out", str(tmp_path), "--max-tokens", "128"],
                         input="\n".join(json.dumps(s) for s in steps) + "\n", text=True,
                         capture_output=True, timeout=600)
    assert out.returncode == 0, out.stderr[-2000:]
    assert [l for l in out.stdout.split("\n") if l.startswith("done")] == ["done 0", "done 1", "done 2"]
    first = torch.from_numpy(np.fromfile(tmp_path / "0.f32", dtype="<f4").reshape(2, -1))
    last = torch.from_numpy(np.fromfile(tmp_path / "2.f32", dtype="<f4").reshape(2, -1))
    assert not (tmp_path / "1.f32").exists()
    assert worst(torch.cat([first, last[1:]]), want[[3, 24, 39]]) < F32_BOUND
    assert worst(last[:1], want_other[[10]]) < F32_BOUND
    gen = subprocess.run([sys.executable, "-m", "zig_ai_amd", "--model", d, "--dtype", "float32",
                          "--prompt-ids", ",".join(map(str, prompt[:9])), "-n", "5",
                          "--temperature", "0", "--json"], cwd=root, text=True, capture_output=True,
                         timeout=600)
    assert gen.returncode == 0, gen.stderr[-2000:]
    outputs = json.loads(gen.stdout.strip().split("\n")[-1])["outputs"]
    assert len(outputs) == 1 and len(outputs[0]) == 5
    logits = plain.forward(cfg, tensors, prompt[:9] + outputs[0])
    for j, tok in enumerate(outputs[0]):
        row = logits[9 + j - 1]
        assert float(row.max() - row[tok]) <= 1e-3 * float(row.abs().max()), (j, tok)


# ------------------------------------------------------------------ kernels alone
def _route_plain(logits, correction, router):
    n = logits.shape[1]
    t = {"x.router": torch.eye(n, dtype=torch.float64), "x.correction": correction}
    return plain.route(logits.double(), t, "x.", router)


@pytest.mark.parametrize("n,top,groups,scale", [(12, 3, (4, 2), 1.5), (16, 4, (4, 3), 2.0),
                                                (7, 7, None, 1.0), (6, 1, (6, 1), 0.5),
                                                (64, 6, (8, 3), 1.0), (9, 2, (1, 1), 1.0),
                                                (300, 8, (10, 4), 2.5)])
def test_router_kernel(n, top, groups, scale):
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(n + top)
    T = 200
    # a few extra columns behind the router's outputs, as the shared expert's gate is
    logits = torch.randn(T, n + 3, generator=g) * 2.0
    router = {"top": top, "scale": scale}
    if groups:
        router["groups"] = {"count": groups[0], "keep": groups[1]}
    # corrections that push every choice score below zero in half of the cases: an output
    # that may not be chosen counts as minus infinity, not as zero
    for shift in (0.0, -3.0):
        correction = torch.randn(n, generator=g) * 0.2 + shift
        chosen, weight = ops.route_topk(logits.to(dev), n, top, correction.to(dev),
                                        groups[0] if groups else 0, groups[1] if groups else 0,
                                        scale, "softmax", False)
        want_c, want_w = _route_plain(logits[:, :n], correction.double(), router)
        got = {(t, int(e)): float(w) for t in range(T)
               for e, w in zip(chosen[t].cpu(), weight[t].cpu())}
        assert len(got) == T * top                      # a row's experts differ
        for t in range(T):
            for e, w in zip(want_c[t].tolist(), want_w[t].tolist()):
                assert (t, e) in got, (t, e, shift)
                assert abs(got[(t, e)] - w) < 1e-6 + 1e-5 * abs(w)


def _latent_attention_case(dtype, H, W, R, requests, page_size, per_item, seed):
    """A paged cache of rows ``[latent | rotated part]`` for ``requests`` = [(cached, new)],
    folded queries for the new tokens, the step's arrays, and what the attention should give
    (float64, with a sink a head)."""
    g = torch.Generator().manual_seed(seed)
    n_pages = sum(-(-(c + n) // page_size) for c, n in requests) + 3
    order = torch.randperm(n_pages, generator=g).tolist()
    plane = torch.zeros(n_pages, 1, page_size, W)
    most = max(-(-(c + n) // page_size) for c, n in requests)
    table = torch.full((len(requests), most + 1), -1, dtype=torch.int32)
    scale = 1.7 * W ** -0.5
    sink = torch.randn(H, generator=g) * 1.5
    qs, positions, items, want = [], [], [], []
    row = 0
    for s, (cached, new) in enumerate(requests):
        keys = (torch.randn(cached + new, W, generator=g)).to(dtype).float()
        for p in range(-(-(cached + new) // page_size)):
            page = order.pop()
            table[s, p] = page
            chunk = keys[p * page_size:(p + 1) * page_size]
            plane[page, 0, :chunk.shape[0]] = chunk
        q = torch.randn(new, H, W, generator=g).to(dtype).float()
        qs.append(q)
        positions += list(range(cached, cached + new))
        for a in range(0, new, per_item):
            items.append((s, row + a, min(per_item, new - a)))
        row += new
        for i in range(new):
            k = keys[:cached + i + 1].double()
            sc = torch.einsum("hw,jw->hj", q[i].double(), k) * scale
            top = torch.maximum(sc.max(dim=1, keepdim=True).values, sink.double()[:, None])
            e = torch.exp(sc - top)
            pr = e / (e.sum(dim=1, keepdim=True) + torch.exp(sink.double()[:, None] - top))
            want.append(pr @ k[:, :R])
    dev = torch.device("cuda")
    mk = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    return (torch.cat(qs).to(dtype).to(dev), plane.to(dtype).to(dev), table.to(dev), mk(positions),
            mk([i[0] for i in items]), mk([i[1] for i in items]), mk([i[2] for i in items]),
            len(items), scale, sink.to(dev), torch.stack(want))


@pytest.mark.parametrize("H,W,R,page_size", [(3, 40, 32, 4), (16, 576, 512, 16), (8, 160, 128, 16),
                                             (4, 96, 96, 16), (5, 48, 24, 8), (40, 80, 72, 16),
                                             (1, 264, 256, 32)])
def test_latent_attention_kernels(H, W, R, page_size):
    from zig_ai_amd.kernels import ops
    # prompt portions behind cached tokens, a first portion, single tokens, one token alone
    requests = [(70, 9), (0, 45), (133, 1), (0, 1), (31, 2)]
    for dtype, waves_list in ((torch.float32, (0,)), (torch.bfloat16, (0, 4))):
        for waves in waves_list:
            most = ops.LATENT_MFMA_ROWS if waves else ops.LATENT_MAX_ROWS
            per_item = max(1, most // min(H, most))
            q, plane, table, pos, iseq, irow, icnt, n, scale, sink, want = _latent_attention_case(
                dtype, H, W, R, requests, page_size, per_item, seed=H + W)
            for keys, nsplit in ((0, 1), (64, 3)):
                got = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink,
                                           keys, nsplit, waves).cpu().double()
                tol = 2e-5 if dtype == torch.float32 else 2e-2
                assert float((got - want).abs().max()) < tol, (dtype, waves, nsplit)
    # single tokens only: a wave a workgroup
    requests = [(200, 1), (0, 1), (63, 1), (64, 1)]
    q, plane, table, pos, iseq, irow, icnt, n, scale, sink, want = _latent_attention_case(
        torch.bfloat16, H, W, R, requests, page_size, 1, seed=7)
    for keys, nsplit in ((0, 1), (64, 4), (128, 2)):
        got = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink, keys,
                                   nsplit, 1).cpu().double()
        assert float((got - want).abs().max()) < 2e-2, nsplit


@pytest.mark.parametrize("H,W,R", [(16, 576, 512), (3, 40, 32)])
def test_latent_decoding_cut_far_beyond_its_contexts(H, W, R):
    """Ranges behind every context, as a recorded step has them: they leave no result, and what their
    places in the workspace held before does not matter (both kernels that merge)."""
    from zig_ai_amd.kernels import ops
    requests = [(200, 1), (0, 1), (63, 1), (64, 1)]
    q, plane, table, pos, iseq, irow, icnt, n, scale, sink, want = _latent_attention_case(
        torch.bfloat16, H, W, R, requests, 16, 1, seed=8)
    few = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink, 64, 4, 1)
    assert float((few.cpu().double() - want).abs().max()) < 2e-2
    for nsplit in (16, 64, 70):
        held = torch.full((4 * H * nsplit * R,), float("nan"), device="cuda")
        del held                                     # (the next tensors of its size lie there)
        many = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink, 64, nsplit, 1)
        if nsplit <= 64:
            assert torch.equal(many, few), nsplit
        assert float((many.cpu().double() - want).abs().max()) < 2e-2, nsplit


@pytest.mark.parametrize("H,R,rotated,page_size", [
    (16, 512, 64, 16), (16, 512, 32, 64), (3, 512, 0, 16), (70, 256, 64, 8), (5, 256, 32, 16), (64, 256, 0, 4),
    (1, 128, 64, 16), (9, 128, 32, 32), (40, 128, 0, 16), (2, 512, 64, 12)])
def test_latent_prefill_on_whole_tiles(H, R, rotated, page_size):
    """Rows that the tiled kernel takes (the last: a page size that it leaves to the other)."""
    from zig_ai_amd.kernels import ops
    requests = [(70, 9), (0, 150), (133, 1), (0, 1), (31, 34), (64, 64), (63, 2), (191, 1)]
    W, most = R + rotated, ops.LATENT_MFMA_ROWS
    q, plane, table, pos, iseq, irow, icnt, n, scale, sink, want = _latent_attention_case(
        torch.bfloat16, H, W, R, requests, page_size, max(1, most // min(H, most)), seed=H + W)
    for keys, nsplit in ((0, 1), (64, 4), (128, 2)):
        got = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink, keys, nsplit,
                                   4).cpu().double()
        # (the probabilities and the result in bfloat16: 2^-9 of values up to 4 either time)
        assert float((got - want).abs().max()) < 2e-2, nsplit


@pytest.mark.parametrize("H,R,rotated,page_size", [
    (16, 512, 64, 16), (3, 512, 32, 64), (40, 512, 0, 4), (17, 256, 64, 8), (1, 128, 32, 16), (16, 128, 0, 32)])
def test_latent_decoding_on_whole_tiles(H, R, rotated, page_size):
    """Single tokens, 128 keys at a time: contexts at the edges of a wave's 16 keys, of the 32 that a product takes
    and of tiles, whole and in ranges of less, one and several tiles, with and without pages."""
    from zig_ai_amd.kernels import ops
    assert ops.latent_range_fits(R + rotated, R, page_size)
    requests = [(c, 1) for c in (0, 1, 15, 16, 30, 31, 32, 47, 95, 96, 126, 127, 128, 159, 255, 256, 300)]
    W = R + rotated
    q, plane, table, pos, iseq, irow, icnt, n, scale, sink, want = _latent_attention_case(
        torch.bfloat16, H, W, R, requests, page_size, 1, seed=H + W)
    for keys, nsplit in ((0, 1), (64, 5), (128, 3), (256, 2), (384, 1)):
        got = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink, keys if nsplit > 1 else 0,
                                   nsplit, 1).cpu().double()
        # (the probabilities and the result in bfloat16: 2^-9 of values up to 4 either time)
        assert float((got - want).abs().max()) < 2e-2, nsplit
    missing, zeros = table.clone(), table.clone()
    plane = torch.cat([plane, torch.zeros_like(plane[:1])])      # a page of zeros at the end
    missing[:, ::3], zeros[:, ::3] = -1, plane.shape[0] - 1
    for keys, nsplit in ((0, 1), (128, 3)):
        got, want = (ops.latent_attention(q, plane, R, t, pos, iseq, irow, icnt, n, scale, sink, keys, nsplit, 1)
                     for t in (missing, zeros))
        assert torch.equal(got, want), nsplit


@pytest.mark.parametrize("H,R,rotated", [(16, 512, 64), (40, 512, 0), (16, 256, 64), (3, 128, 32)])
def test_latent_decoding_is_off_by_its_results_rounding(H, R, rotated):
    """Single tokens, whole and in ranges: no further from 64 bits than the result's own rounding to bfloat16, but
    for 3 in 100 (scores and weights are rounded far below that)."""
    from zig_ai_amd.kernels import ops
    q, plane, table, pos, iseq, irow, icnt, n, scale, sink, want = _latent_attention_case(
        torch.bfloat16, H, R + rotated, R, [(c, 1) for c in (40, 100, 129, 300, 517, 1000)], 16, 1, seed=H)
    bound = 1.03 * rel_norm(want.bfloat16().double(), want)
    for keys, nsplit in ((0, 1), (128, 8), (512, 2)):
        got = ops.latent_attention(q, plane, R, table, pos, iseq, irow, icnt, n, scale, sink, keys, nsplit, 1).cpu().double()
        off = rel_norm(got, want)
        assert off < bound, nsplit


@pytest.mark.parametrize("R,rotated,page_size", [(512, 64, 16), (256, 32, 4), (128, 0, 64), (512, 64, 12)])
def test_latent_prefill_without_a_page(R, rotated, page_size):
    """A table entry below zero stands for rows of zeros, never for another request's page."""
    from zig_ai_amd.kernels import ops
    H, W, most = 8, R + rotated, ops.LATENT_MFMA_ROWS
    requests = [(70, 9), (0, 150), (133, 1), (200, 31)]
    q, plane, table, pos, iseq, irow, icnt, n, scale, sink, _ = _latent_attention_case(
        torch.bfloat16, H, W, R, requests, page_size, max(1, most // H), seed=W)
    missing = table.clone()
    missing[:, ::3] = -1                             # every third page, the first among them
    plane = torch.cat([plane, torch.zeros_like(plane[:1])])      # a page of zeros at the end
    zeros = table.clone()
    zeros[:, ::3] = plane.shape[0] - 1
    for keys, nsplit in ((0, 1), (64, 4)):
        got, want = (ops.latent_attention(q, plane, R, t, pos, iseq, irow, icnt, n, scale, sink, keys, nsplit, 4)
                     for t in (missing, zeros))
        assert torch.equal(got, want), nsplit


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,N,K,mode", [(3, 24, 16, None), (8, 128, 64, "element"), (5, 40, 32, "head"),
                                        (1, 8, 320, "element"), (40, 72, 8, None)])
def test_head_linear_kernel(dtype, H, N, K, mode):
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(H * N + K)
    T = 37
    x = torch.randn(T, H, K + 8, generator=g).to(dtype)
    w = (torch.randn(H, N, K, generator=g) * K ** -0.5).to(dtype)
    gate = torch.randn(T, 16 + (H if mode == "head" else H * N), generator=g).to(dtype)
    got = ops.head_linear(x.to(dev), 8, w.to(dev), gate=gate.to(dev) if mode else None, gate_col=16,
                          gate_mode=mode).cpu().double()
    want = torch.einsum("thk,hnk->thn", x[:, :, 8:].double(), w.double())
    if mode == "head":
        want = want * torch.sigmoid(gate[:, 16:].double())[:, :, None]
    elif mode == "element":
        want = want * torch.sigmoid(gate[:, 16:].double()).view(T, H, N)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    assert float((got - want).abs().max()) < tol * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("T", [1, 16, 17, 64, 65, 200])
@pytest.mark.parametrize("H,N,K,mode", [(3, 140, 264, "element"), (2, 128, 512, "head"), (5, 70, 128, "element"),
                                        (1, 512, 136, None), (4, 16, 8, None)])
def test_head_linear_at_the_edges_of_its_tiles(T, H, N, K, mode):
    """Rows of decode batches and of tiles, K split or not and off the tiles' 64, columns that do
    and do not fill 16-byte stores, into rows wider than the result."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(T + N + K)
    x = torch.randn(T, H, K + 16, generator=g).bfloat16()
    w = (torch.randn(H, N, K, generator=g) * K ** -0.5).bfloat16()
    gate = torch.randn(T, 4 + (H if mode == "head" else H * N), generator=g).bfloat16()
    for dtype in (torch.bfloat16, torch.float32):
        out = torch.full((T, H, N + 8), 7.0, dtype=dtype, device=dev)
        ops.head_linear(x.to(dev), 8, w.to(dev), out=out, out_col=4, gate=gate.to(dev) if mode else None,
                        gate_col=4, gate_mode=mode)
        want = torch.einsum("thk,hnk->thn", x[:, :, 8:8 + K].double(), w.double())
        if mode == "head":
            want = want * torch.sigmoid(gate[:, 4:].double())[:, :, None]
        elif mode == "element":
            want = want * torch.sigmoid(gate[:, 4:].double()).view(T, H, N)
        got = out.cpu().double()
        # (32-bit sums of K products; one rounding to bfloat16 on the way out)
        bound = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20) * max(1.0, float(want.abs().max()))
        assert float((got[:, :, 4:-4] - want).abs().max()) < bound
        assert bool((got[:, :, :4] == 7).all()) and bool((got[:, :, -4:] == 7).all())


@pytest.mark.parametrize("T", [5, 40])
def test_products_of_views_that_start_off_16_bytes(T):
    """Grouped products and heads' own products take views that start anywhere: the same bits."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(T)

    def shifted(t):
        room = torch.empty(t.numel() + 4, dtype=t.dtype, device=dev)
        room[4:] = t.reshape(-1)
        return room[4:].view(t.shape)                # eight bytes behind the allocation's start

    x = torch.randn(T, 3, 72, generator=g).bfloat16().to(dev)
    w = torch.randn(3, 40, 64, generator=g).bfloat16().to(dev)
    want = ops.head_linear(x, 8, w)
    assert torch.equal(ops.head_linear(shifted(x), 8, w), want)
    assert torch.equal(ops.head_linear(x, 8, shifted(w)), want)
    rows = torch.randn(T, 72, generator=g).bfloat16().to(dev)
    experts = torch.randn(4, 48, 72, generator=g).bfloat16().to(dev)
    chosen = torch.randint(0, 4, (T, 1), generator=g).int().to(dev)
    lists, counts = ops.expert_lists(None, chosen, T, 4)
    want = ops.grouped_linear(rows, experts, lists, counts, T, per_token=True)
    assert torch.equal(ops.grouped_linear(shifted(rows), experts, lists, counts, T, per_token=True), want)
    assert torch.equal(ops.grouped_linear(rows, shifted(experts), lists, counts, T, per_token=True), want)


def test_token_side_kernels():
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(1)
    T, dim, V, width = 19, 12, 50, 40
    gate = torch.randn(T, dim, generator=g) * 2
    table = torch.randn(V, 5 * dim, generator=g)
    ids = torch.randint(0, V, (T,), generator=g, dtype=torch.int32)
    got = ops.table_gate(gate.to(dev), ids.to(dev), table.to(dev), 3 * dim, "gelu_tanh").cpu().double()
    want = plain.gelu_tanh(gate.double()) * table.double()[ids.long()][:, 3 * dim:4 * dim]
    assert float((got - want).abs().max()) < 1e-5
    stream = torch.randn(T, width, generator=g)
    y = torch.randn(T, width, generator=g) * 3
    w = torch.randn(width, generator=g)
    res = stream.to(dev).clone()
    ops.normed_add_(res, y.to(dev), w.to(dev), 1e-3, 0.3)
    want = stream.double() + 0.3 * plain.rms_norm(y.double(), w.double(), 1e-3)
    assert float((res.cpu().double() - want).abs().max()) < 1e-5
    z = torch.randn(T, width, generator=g) * 20
    got = ops.softcap_(z.to(dev).clone(), 7.0).cpu().double()
    assert float((got - 7.0 * torch.tanh(z.double() / 7.0)).abs().max()) < 1e-5


@pytest.mark.parametrize("mode,renorm", [("softmax", False), ("sigmoid", True)])
@pytest.mark.parametrize("n,groups,keep,top", [(1, 0, 0, 1), (30, 0, 0, 4), (32, 4, 2, 4), (64, 16, 3, 7),
                                               (64, 0, 0, 64), (65, 0, 0, 8), (66, 6, 2, 5)])
def test_router_ties_and_values_that_compare_false(n, groups, keep, top, mode, renorm):
    """One output a lane or more of them: of equal scores the lower index first, an output whose
    score is NaN last of all (and output 0 where nothing is left)."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(n + top)
    T = 24
    logits = torch.randint(-2, 3, (T, n), generator=g).float()          # ties
    correction = torch.zeros(n)
    if n > top + 2 and not groups:
        correction[1] = float("nan")
    chosen, weight = ops.route_topk(logits.to(dev), n, top, correction.to(dev), groups, keep, 1.5, mode, renorm)
    s = torch.softmax(logits.double(), 1) if mode == "softmax" else torch.sigmoid(logits.double())
    for t in range(T):
        # (whole numbers stand for the scores, which rise with them: the kernel's ties are exact)
        c = [float(v) if not math.isnan(float(k)) else None for v, k in zip(logits[t], correction)]
        usable = [e for e in range(n) if c[e] is not None]
        if groups and keep < groups:
            per = n // groups
            best = sorted(range(groups), key=lambda q: (-max(c[q * per:(q + 1) * per]), q))[:keep]
            usable = [e for e in usable if e // per in best]
        want = sorted(usable, key=lambda e: (-c[e], e))[:top]
        assert chosen[t].tolist() == want
        w = s[t][want]
        w = w / w.sum() * 1.5 if renorm else w * 1.5
        assert float((weight[t].cpu().double() - w).abs().max()) < 1e-6
    nothing = torch.full((n,), float("nan"))
    chosen, _ = ops.route_topk(logits.to(dev), n, top, nothing.to(dev), 0, 0, 1.0, mode, renorm)
    assert not bool(chosen.any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Rq,R,Dr,rot,adjacent", [(1536, 512, 64, 64, True), (2048, 512, 32, 16, False), (40, 24, 8, 8, True),
                                                  (300, 257, 0, 0, False), (2056, 64, 16, 16, True), (64, 520, 8, 0, False)])
def test_latent_prepare_kernels(dtype, Rq, R, Dr, rot, adjacent):
    """Latents that a workgroup holds in registers and longer ones."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(Rq + R)
    T, page, c_col = 5, 4, Rq + 8
    down = torch.randn(T, c_col + R + Dr, generator=g).to(dtype)
    qw, cw = torch.randn(Rq, generator=g), torch.randn(R, generator=g)
    positions, slots = [0, 3, 7, 100, 2000], [2, 9, -1, 0, 7]
    freq = 1e4 ** (-torch.arange(max(1, rot // 2)).float() / max(1, rot // 2))
    plane = torch.full((3, 1, page, R + Dr), 9.0, dtype=dtype, device=dev)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    cq = ops.latent_prepare(down.to(dev), 0, Rq, c_col, R, Dr, qw.to(dev), cw.to(dev), 1e-6, i32(positions),
                            i32(slots), freq.to(dev) if rot else None, rot, adjacent, plane, 1.25)
    x = down.double()
    tol = 2e-5 if dtype == torch.float32 else 2e-2      # (32-bit angles up to 2,000; one rounding of values up to 5)
    norm = lambda v, w: v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-6) * w.double()
    want = norm(x[:, :Rq], qw)
    assert float(((cq.cpu().double() - want) / (1 + want.abs())).abs().max()) < tol
    c, kr = norm(x[:, c_col:c_col + R], cw), x[:, c_col + R:].clone()
    if rot:
        half = rot // 2
        angle = (torch.tensor(positions).float()[:, None] * freq[None]).double()
        a = torch.arange(half) * 2 if adjacent else torch.arange(half)
        b = a + 1 if adjacent else a + half
        u, v = kr[:, a].clone(), kr[:, b].clone()
        kr[:, a] = (u * torch.cos(angle) - v * torch.sin(angle)) * 1.25
        kr[:, b] = (v * torch.cos(angle) + u * torch.sin(angle)) * 1.25
    got, rows = plane.cpu().double().view(-1, R + Dr), torch.cat([c, kr], 1)
    for t, s in enumerate(slots):
        if s >= 0:
            assert float(((got[s] - rows[t]) / (1 + rows[t].abs())).abs().max()) < tol
    untouched = [s for s in range(12) if s not in slots]
    assert bool((got[untouched] == 9).all())


@pytest.mark.parametrize("H,rotated,mode,lens,ctxs", [
    (16, 64, None, [33, 64, 65], [0, 0, 0]), (3, 64, "element", [2, 129, 200], [0, 77, 5]),
    (5, 0, "head", [63, 300], [1, 640]), (1, 64, "head", [2], [0]), (40, 0, None, [900], [0])])
def test_latent_attention_over_formed_keys(H, rotated, mode, lens, ctxs):
    """Portions at the edges of items of 64 rows and of tiles of 64 keys, with and without cached rows, from one
    workgroup to several rounds of them: rows laid out, queries turned, keys and values formed, attention,
    sink and gate."""
    from zig_ai_amd.engine.batch import _make_items
    from zig_ai_amd.kernels import ops
    dev, R, d, page = torch.device("cuda"), 256, 128, 12
    g = torch.Generator().manual_seed(H + sum(lens))
    S, T, W = len(lens), sum(lens), R + rotated
    pages = [-(-(n + c) // page) for n, c in zip(lens, ctxs)]
    table = torch.full((S, max(pages) + 1), -1, dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=g), 0
    for s, n in enumerate(pages):
        table[s, :n] = order[at:at + n]
        at += n
    plane = torch.randn(sum(pages), 1, page, W, generator=g).bfloat16()
    q = torch.randn(T, H, d + rotated, generator=g).bfloat16()
    up = (torch.randn(2 * H * d, R, generator=g) * R ** -0.5).bfloat16()
    rot_dims = rotated // 2
    inv = torch.rand(max(rot_dims // 2, 1), generator=g) if rot_dims else None
    sink = torch.randn(H, generator=g)
    gate = torch.randn(T, 8 + (H * d if mode == "element" else -(-H // 8) * 8), generator=g).bfloat16()
    positions = [c + j for n, c in zip(lens, ctxs) for j in range(n)]
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    seq, row0, cnt = _make_items(lens, ops.LATENT_EXPANDED_ROWS, 2)
    start = [sum(lens[:s]) for s in range(S + 1)]
    turned = q.to(dev)
    latent, rot = ops.latent_open_rows(turned, d, rotated, mk(positions), inv.to(dev) if rot_dims else None, rot_dims,
                                       True, 1.25, plane.to(dev), R, table.to(dev), mk(start), mk(ctxs),
                                       T + sum(ctxs))
    kv = ops.linear(latent, up.to(dev))
    got = ops.latent_expanded(turned, kv, rot, mk(positions), (mk(seq), mk(row0), mk(cnt), len(seq)), mk(start),
                              mk(ctxs), 0.09, sink.to(dev), gate.to(dev) if mode else None, 8, mode).cpu().double()
    qd = q.double()
    if rot_dims:
        angle = torch.tensor(positions).double()[:, None, None] * inv.double()
        c, s = 1.25 * angle.cos(), 1.25 * angle.sin()
        u, v = qd[..., d:d + rot_dims:2].clone(), qd[..., d + 1:d + rot_dims:2].clone()
        qd[..., d:d + rot_dims:2], qd[..., d + 1:d + rot_dims:2] = u * c - v * s, v * c + u * s
    for s in range(S):
        n = lens[s] + ctxs[s]
        rows = plane[table[s, :pages[s]].long()].view(-1, W)[:n]
        at = start[s] + sum(ctxs[:s])
        assert torch.equal(latent[at:at + n].cpu(), rows[:, :R])
        assert not rotated or torch.equal(rot[at:at + n].cpu(), rows[:, R:])
        formed = (rows[:, :R].double() @ up.double().T).view(n, 2, H, d)
        keys = torch.cat([formed[:, 0], rows[:, None, R:].double().expand(n, H, rotated)], dim=2)
        mine = slice(start[s], start[s + 1])
        scores = torch.einsum("thd,nhd->htn", qd[mine], keys) * 0.09
        scores = scores.masked_fill(torch.arange(n)[None, :] > torch.tensor(positions[mine])[:, None], -math.inf)
        weights = torch.softmax(torch.cat([scores, sink.double()[:, None, None].expand(H, lens[s], 1)], dim=2), dim=2)
        want = torch.einsum("htn,nhd->thd", weights[..., :n], formed[:, 1])
        if mode:
            z = torch.sigmoid(gate[mine, 8:].double())
            want = want * (z[:, :H, None] if mode == "head" else z.view(-1, H, d))
        # (roundings to bfloat16, 2^-9 at most and a third of its square on average, of queries' turned parts, keys,
        # values, weights and the result: sqrt(5 / 3) 2^-9 = 2.5e-3 of the norm; scores of deviation 1.2)
        assert rel_norm(got[mine], want) < 5e-3, s


@pytest.mark.parametrize("tokens,behind", [(16, 0), (64, 0), (130, 0), (300, 0), (16, 128), (40, 600), (1000, 0)])
def test_formed_keys_are_as_exact_as_folded_queries(tokens, behind):
    """The error against 64 bits of attention over formed keys and values is no larger than the folded kernels' on
    the same rows (both round as many values to bfloat16; over 8 drawings the two come within 1 in 100 of each
    other when the roundings alone are worked out)."""
    from zig_ai_amd.engine.batch import _make_items
    from zig_ai_amd.kernels import ops
    dev, H, R, d, rotated, page = torch.device("cuda"), 8, 512, 128, 64, 16
    n, W, scale = tokens + behind, R + rotated, (d + rotated) ** -0.5
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    table, positions = mk(range(-(-n // page))).view(1, -1), mk(range(behind, n))
    start, context = mk([0, tokens]), mk([behind])

    def items(rows):
        seq, row0, count = _make_items([tokens], rows, 2)
        return mk(seq), mk(row0), mk(count), len(seq)

    off = {"folded": 0.0, "formed": 0.0}
    for seed in range(8):
        g = torch.Generator(device=dev).manual_seed(seed)
        rand = lambda *shape: torch.randn(*shape, device=dev, generator=g)
        up = (rand(2, H * d, R) * R ** -0.5).bfloat16()
        plane, q = rand(table.shape[1], 1, page, W).bfloat16(), rand(tokens, H, d + rotated).bfloat16()
        inv = torch.tensor([1e4 ** (-i / 32) for i in range(32)], device=dev)
        rows = plane.view(-1, W)[:n].double()
        keys, values = ((rows[:, :R] @ w.double().T).view(n, H, d) for w in up)
        angle = positions.double()[:, None, None] * inv.double()
        u, v = q[..., d:d + 32].double(), q[..., d + 32:].double()
        turned = torch.cat([q[..., :d].double(), u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()], 2)
        keys = torch.cat([keys, rows[:, None, R:].expand(n, H, rotated)], 2)
        want = torch.empty(tokens, H, d, dtype=torch.float64, device=dev)
        for h in range(H):
            s = (turned[:, h] @ keys[:, h].T.contiguous()) * scale
            s = s.masked_fill(torch.arange(n, device=dev)[None] > positions[:, None], -math.inf)
            want[:, h] = s.softmax(1) @ values[:, h].contiguous()
        fold = up[0].view(H, d, R).transpose(1, 2).contiguous()
        qf = ops.latent_fold(q, fold, rotated, positions, inv, rotated, False)
        o = ops.latent_attention(qf, plane, R, table, positions, *items(64 // H), scale, None, 0, 1, 4)
        folded = ops.head_linear(o, 0, up[1].view(H, d, R))
        latent, rot = ops.latent_open_rows(q, d, rotated, positions, inv, rotated, False, 1.0, plane, R, table, start,
                                           context, n)
        kv = ops.linear(latent, up.view(2 * H * d, R))
        formed = ops.latent_expanded(q, kv, rot, positions, items(64), start, context, scale)
        for name, got in (("folded", folded), ("formed", formed)):
            off[name] += rel_norm(got.double(), want) / 8
    assert off["formed"] < 1.015 * off["folded"], off


@pytest.mark.parametrize("T", [1, 7, 16, 17])
@pytest.mark.parametrize("H,R,d,rotated,rot_dims,adjacent", [(16, 512, 128, 64, 64, True), (3, 40, 24, 16, 8, False),
                                                             (5, 72, 128, 32, 0, True), (2, 128, 264, 64, 64, False)])
def test_latent_fold_in_one_launch(T, H, R, d, rotated, rot_dims, adjacent):
    """A decode batch's folded queries against the product and the rotation one after the other: the same bits
    (17 rows, and heads whose K is shared out, take the two)."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(T + H + d)
    q = torch.randn(T, H, d + rotated, generator=g).bfloat16().to(dev)
    fold = (torch.randn(H, R, d, generator=g) * d ** -0.5).bfloat16().to(dev)
    positions = torch.randint(0, 100000, (T,), generator=g, dtype=torch.int32).to(dev)
    inv = torch.rand(max(rot_dims // 2, 1), generator=g).to(dev) if rot_dims else None
    got = ops.latent_fold(q, fold, rotated, positions, inv, rot_dims, adjacent, 1.25)
    want = torch.full((T, H, R + rotated), float("nan"), dtype=torch.bfloat16, device=dev)
    ops.head_linear(q, 0, fold, out=want, out_col=0)
    ops.rotate_part_(q, d, want, R, rotated, positions, inv, rot_dims, adjacent, 1.25)
    assert torch.equal(got, want)


@pytest.mark.parametrize("T,K,dim", [(1, 8, 5), (3, 250 * 8, 40), (16, 2048, 256), (8, 4104, 17), (17, 64, 32),
                                     (8, 4096, 17), (1, 6144, 24), (9, 4096, 32), (2, 2560, 32)])
@pytest.mark.parametrize("table_dtype", [torch.float32, torch.bfloat16])
def test_table_gate_on_its_own_product(T, K, dim, table_dtype):
    """Steps of K below, at and beyond what eight waves have under way; outputs that fill no tile; ids that are not in
    the table."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(T + K + dim)
    x = torch.randn(T, K, generator=g).bfloat16()
    w = (torch.randn(dim, K, generator=g) * K ** -0.5).bfloat16()
    table = torch.randn(50, dim + 9, generator=g).to(table_dtype)
    ids = torch.randint(0, 50, (T,), generator=g, dtype=torch.int32)
    ids[0] = 50 if T > 1 else 3
    ops.form_log = []
    try:
        got = ops.table_gate_linear(x.to(dev), w.to(dev), ids.to(dev), table.to(dev), 9, "gelu_tanh").cpu().double()
        product, = [r for r in ops.form_log if r["op"] == "linear"]
    finally:
        ops.form_log = None
    assert (product["M"], product["N"], product["K"]) == (T, dim, K)
    assert (product.get("kernel") == "table_gate") == ops.table_gate_fuses(T, K)
    rows = torch.where((ids < 50)[:, None], table[ids.clamp(max=49).long(), 9:].double(), torch.zeros(()).double())
    want = torch.nn.functional.gelu(x.double() @ w.double().T, approximate="tanh") * rows
    # (product and result are rounded to bfloat16: 2^-9 each of values that the gate carries on with slopes up to 1.13)
    assert rel_norm(got, want) < 2.0 ** -7
    assert T == 1 or float(got[0].abs().max()) == 0.0


def rel_norm(got, want):
    return float((got - want).norm() / want.norm())
