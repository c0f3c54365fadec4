"""Rudilix through the engine against the plain implementation (``plain_rudilix.py``,
float64, whole sequences, one function per mechanism).

float32 runs are held to the plain logits row by row (root mean square of the
difference over the vocabulary, relative to the logits' own spread): measured 1e-6 to
7e-6, bound 1e-4.  That is the bound that can fail, and every schedule, cut and batch is
held to it.  A bfloat16 run is chaotic at single rows: the delta rule's read-out is divided
by its own root mean square, which for a request's first tokens is a multiple of q . k, a
number that may be as small as its rounding error, and the weights here are drawn sharp on
purpose.  So bfloat16 rows are held to the plain logits by their median and their ninth
decile, and the worst row only to a bound that says that nothing is grossly wrong; the
bounds were measured first (median 0.009 to 0.011, ninth decile 0.015 to 0.02, worst row
0.07 and 0.28) and then set with margins.  How a bfloat16 request was cut and batched must
not show beyond rounding either: every schedule is held to the whole prompts' run."""

import math

import pytest
import torch

import engine_util as eu
import plain_rudilix as plain
import rudilix_util as ru

pytestmark = pytest.mark.gpu

F32_BOUND = 1e-4
BF16_MEDIAN, BF16_DECILE, BF16_WORST = 0.04, 0.12, 0.6
BF16_BETWEEN_MEDIAN, BF16_BETWEEN_WORST = 1e-3, 0.03      # one schedule against another (measured 0 and 0.006)


def build(cfg, seed=0, dtype="float32", tensors=None):
    from zig_ai_amd.engine import DecoderModel
    d, tensors = ru.folder(cfg, seed, tensors)
    return DecoderModel.from_folder(d, dtype), tensors


def runner_for(model, page_size=4, tokens=256, slots=4, graphs=True):
    from zig_ai_amd.engine import ModelRunner
    return ModelRunner(model, page_size=page_size, num_pages=max(1, -(-tokens // page_size)),
                       num_slots=slots, use_graphs=graphs)


def plain_logits(cfg, tensors, prompts):
    return [plain.forward(cfg, tensors, p).float() for p in prompts]


def worst(got, want):
    return float(ru.row_error(got, want).max())


def assert_bfloat16_close(got, want, what=None):
    e = ru.row_error(got, want)
    found = (float(e.median()), float(e.quantile(0.9)), float(e.max()))
    assert found[0] < BF16_MEDIAN and found[1] < BF16_DECILE and found[2] < BF16_WORST, (what, found)


# ----------------------------------------------------------- each mechanism alone
ALONE = {
    "ssd": ru.one_layer("mamba2", ru.ssd()),
    "ssd one group": ru.one_layer("mamba2", ru.ssd(heads=2, vdim=24, state=72, groups=1,
                                                     norm_groups=1, conv=2), ff=0),
    "delta": ru.one_layer("channel_delta", ru.delta()),
    "delta wide": ru.one_layer("channel_delta", ru.delta(heads=2, kv_heads=1, dim=40, vdim=72,
                                                          conv=4), ff=0),
    "delta one tap": ru.one_layer("channel_delta", ru.delta(heads=3, kv_heads=3, dim=16, vdim=16,
                                                             conv=1)),
    "attention + delta": ru.one_layer("parallel", ru.parallel()),
    "attention alone": ru.one_layer("parallel", ru.parallel(right_scale=0.0), ff=0),
    "attention, full rotation, no window": ru.one_layer("parallel", ru.parallel(
        ru.attention(heads=6, kv_heads=2, dim=16, vdim=16, window=0, rot_dims=16, scale=0.4),
        right_scale=0.0)),
}


@pytest.mark.parametrize("name", sorted(ALONE))
def test_mechanism_alone(name):
    cfg = ALONE[name]
    model, tensors = build(cfg, seed=3)
    prompts = [ru.tokens(70, cfg["vocab"], 1), ru.tokens(5, cfg["vocab"], 2)]
    want = plain_logits(cfg, tensors, prompts)
    runner = runner_for(model)
    got = eu.run_schedule(runner, prompts, eu.whole([len(p) for p in prompts]))
    for g, w in zip(got, want):
        assert worst(g, w) < F32_BOUND
    # the same, token by token from the first token on: the state and the cache alone
    got = eu.run_schedule(runner, prompts, eu.bulk_then_single([len(p) for p in prompts], tail=10 ** 6))
    for g, w in zip(got, want):
        assert worst(g, w) < F32_BOUND


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
    cfg = ru.TINY_ALL if which == "all" else ru.TINY_OTHER
    model, tensors = build(cfg, seed=11)
    prompts = [ru.tokens(n, cfg["vocab"], 20 + i) for i, n in enumerate(LENGTHS)]
    want = plain_logits(cfg, tensors, prompts)
    for name, schedule in schedules(LENGTHS).items():
        # a pool for the most tokens live at any time: pages and slots are used again
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
    cfg = ru.TINY_ALL if which == "all" else ru.TINY_OTHER
    model, tensors = build(cfg, seed=11, dtype="bfloat16")
    prompts = [ru.tokens(n, cfg["vocab"], 20 + i) for i, n in enumerate(LENGTHS)]
    want = plain_logits(cfg, tensors, prompts)
    base = None
    for name, schedule in schedules(LENGTHS).items():
        peak = eu.peak_tokens(LENGTHS, schedule, round_to=16)
        runner = runner_for(model, page_size=16, tokens=peak, slots=4)
        got = eu.run_schedule(runner, prompts, schedule)
        assert_bfloat16_close(torch.cat(got), torch.cat(want), name)
        if base is None:
            base = got
        e = ru.row_error(torch.cat(got), torch.cat(base))
        assert float(e.median()) < BF16_BETWEEN_MEDIAN and float(e.max()) < BF16_BETWEEN_WORST, \
            (name, float(e.median()), float(e.max()))


# ---------------------------------------- configurations drawn at random, both types
@pytest.mark.parametrize("seed", range(12))
def test_random_configurations(seed):
    cfg = ru.random_config(seed)
    lengths = [70, 1, 33, 12, 2]
    prompts = [ru.tokens(n, cfg["vocab"], 90 + i) for i, n in enumerate(lengths)]
    model, tensors = build(cfg, seed=seed)
    want = plain_logits(cfg, tensors, prompts)
    for name, schedule in (("whole", eu.whole(lengths)),
                           ("portions", eu.changing_portions(lengths, seed=seed)),
                           ("mixed", eu.mixed(lengths, seed=seed, max_live=3, decode_tail=9))):
        peak = eu.peak_tokens(lengths, schedule, round_to=16)
        runner = runner_for(model, page_size=4 if seed % 2 else 16, tokens=peak, slots=3)
        got = eu.run_schedule(runner, prompts, schedule)
        # (a model drawn with hardly any spread in its logits is measured against that
        # spread all the same; the bound allows for it)
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
        e = ru.row_error(torch.cat(got), torch.cat(base))
        assert float(e.median()) < BF16_BETWEEN_MEDIAN, float(e.median())


# --------------------------------------------- window edges, with scores that stand out
def sharp_window_cfg(window, rot):
    # a scale that makes the softmax all but choose one key: a key wrongly seen or wrongly
    # hidden then takes or loses nearly all of a query's weight
    att = ru.attention(heads=2, kv_heads=1, dim=16, vdim=16, window=window, rot_dims=rot,
                       base=100.0, scale=2.5)
    return ru.one_layer("parallel", ru.parallel(att, left_scale=1.0, right_scale=0.0), ff=0)


@pytest.mark.parametrize("window,rot", [(7, 0), (16, 8), (1, 16), (21, 4)])
def test_window_edges(window, rot):
    cfg = sharp_window_cfg(window, rot)
    model, tensors = build(cfg, seed=5)
    n = 90
    prompts = [ru.tokens(n, cfg["vocab"], 7)]
    want = plain_logits(cfg, tensors, prompts)[0]
    # the test can see an edge that is one token off: the plain implementation itself,
    # one key more or one fewer, is far from what it gives with the right window
    for other in (window - 1, window + 1):
        if other >= 1:
            off = sharp_window_cfg(other, rot)
            assert worst(plain.forward(off, tensors, prompts[0]).float(), want) > 0.05
    for page_size in (4, 16):
        for name, schedule in (("whole", eu.whole([n])),
                               ("decoded", eu.bulk_then_single([n], tail=n - 3)),
                               ("portions", eu.changing_portions([n], sizes=(5, 2, window, 3, window + 1)))):
            runner = runner_for(model, page_size=page_size, tokens=128)
            got = eu.run_schedule(runner, prompts, schedule)[0]
            assert worst(got, want) < 2e-3, (name, page_size)


# ------------------- key and value widths that the matrix-core attention kernels take
@pytest.mark.parametrize("dim,window,rot", [(64, 40, 32), (128, 0, 128), (64, 130, 0)])
def test_matrix_core_attention_with_gate(dim, window, rot):
    att = ru.attention(heads=4, kv_heads=2, dim=dim, vdim=dim, window=window, rot_dims=rot,
                       base=1000.0, scale=dim ** -0.5)
    cfg = ru.config([ru.layer("parallel", ru.parallel(att, ru.delta(), 1.0, 0.5), ff=64)], width=128)
    model, tensors = build(cfg, seed=6, dtype="bfloat16")
    assert model.blocks[0].parts["left"].mfma
    lengths = [200, 70, 3]
    prompts = [ru.tokens(n, cfg["vocab"], 50 + i) for i, n in enumerate(lengths)]
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
        e = ru.row_error(torch.cat(got), torch.cat(base))
        assert float(e.median()) < BF16_BETWEEN_MEDIAN and float(e.max()) < BF16_BETWEEN_WORST, \
            (name, float(e.median()), float(e.max()))


# ---------------- a width at which a decode batch's opening products run the norm themselves
def test_decode_batches_at_a_width_of_512():
    from zig_ai_amd.kernels import ops
    cfg = ru.config([ru.layer("parallel", ru.parallel()), ru.layer("mamba2", ru.ssd()),
                     ru.layer("channel_delta", ru.delta(), ff=0)], width=512)
    model, tensors = build(cfg, seed=13, dtype="bfloat16")
    assert ops.normed_rows_fusable(3, 512)
    lengths = [60, 25, 8]
    prompts = [ru.tokens(n, cfg["vocab"], 70 + i) for i, n in enumerate(lengths)]
    want = plain_logits(cfg, tensors, prompts)
    whole = eu.run_schedule(runner_for(model, page_size=16, tokens=256), prompts, eu.whole(lengths))
    # all three decode together from their fifth token on: steps of three rows
    steps = [([(i, 0, 4) for i in range(3)], [])]
    steps += [([(i, p, p + 1) for i, n in enumerate(lengths) if p < n],
               [i for i, n in enumerate(lengths) if p == n - 1]) for p in range(4, max(lengths))]
    got = eu.run_schedule(runner_for(model, page_size=16, tokens=256, graphs=False), prompts, steps)
    # (such a step does take that form)
    from zig_ai_amd.engine import StepEntry
    runner = runner_for(model, page_size=16, tokens=64, graphs=False)
    runner.admit("x")
    runner.step([StepEntry("x", prompts[2][:4], [])])
    ops.form_log = []
    try:
        runner.step([StepEntry("x", prompts[2][4:5], [0])])
        assert any(r.get("norm_in_product") for r in ops.form_log if r["op"] == "linear")
    finally:
        ops.form_log = None
    assert_bfloat16_close(torch.cat(got), torch.cat(want))
    # (a product that runs the norm rounds x * weight and scales its sums, the norm as a
    # kernel rounds x * scale * weight: the two runs differ as two roundings do, measured
    # median 0.010, worst 0.038)
    assert_bfloat16_close(torch.cat(got), torch.cat(whole))
    # and replayed from graphs
    again = eu.run_schedule(runner_for(model, page_size=16, tokens=256), prompts, steps)
    e = ru.row_error(torch.cat(again), torch.cat(got))
    assert float(e.max()) < BF16_BETWEEN_WORST


# ----------------------------------------------------------------- far tokens count
@pytest.mark.parametrize("kind", ["mamba2", "channel_delta"])
def test_far_tokens_reach_the_end(kind):
    mixer = ru.ssd(heads=2, vdim=16, state=16, groups=1, norm_groups=1, conv=2) \
        if kind == "mamba2" else ru.delta(heads=2, kv_heads=2, dim=16, vdim=16, conv=2)
    cfg = ru.one_layer(kind, mixer, ff=0)
    tensors = ru.make_tensors(cfg, seed=9)
    tensors["l0.mix.A_log"] = torch.full_like(tensors["l0.mix.A_log"], -8.0)   # all but no decay
    model, tensors = build(cfg, tensors=tensors)
    # (the delta rule overwrites: its state of 16 key channels keeps a token for some tens of
    # steps whatever the decay)
    n = 400 if kind == "mamba2" else 40
    a = ru.tokens(n, cfg["vocab"], 3)
    b = list(a)
    b[1] = (b[1] + 1) % cfg["vocab"]
    wa, wb = plain.forward(cfg, tensors, a).float(), plain.forward(cfg, tensors, b).float()
    assert worst(wb[-8:], wa[-8:]) > 1e-2          # the second token still shows at the end
    for prompt, want in ((a, wa), (b, wb)):
        for schedule in (eu.whole([n]), eu.bulk_then_single([n], tail=64),
                         eu.changing_portions([n], sizes=(33, 2, 64, 17))):
            got = eu.run_schedule(runner_for(model, tokens=512), [prompt], schedule)[0]
            assert worst(got, want) < F32_BOUND
    # nothing is left of a request whose slot is taken again: b after a in a pool of one slot
    runner = runner_for(model, tokens=512, slots=1)
    for prompt, want in ((a, wa), (b, wb), (a, wa)):
        got = eu.run_schedule(runner, [prompt], eu.bulk_then_single([n], tail=5))[0]
        assert worst(got, want) < F32_BOUND


# ------------------------------------- a long context cut into ranges, with the gate
def test_long_context_without_window():
    cfg = ru.TINY_OTHER
    model, tensors = build(cfg, seed=4)
    n = 700
    prompts = [ru.tokens(n, cfg["vocab"], 1), ru.tokens(30, cfg["vocab"], 2)]
    want = plain_logits(cfg, tensors, prompts)
    runner = runner_for(model, page_size=16, tokens=1024)
    wants = [list(range(n - 90, n)), list(range(30))]
    steps = [([(0, 0, n - 80)], [])]
    # the long request decodes beside the short one's portions and single tokens
    steps += [([(0, n - 80 + i, n - 79 + i)] + ([(1, 3 * i, 3 * i + 3)] if i < 10 else []),
               [1] if i == 9 else []) for i in range(80)]
    steps[-1] = (steps[-1][0], [0])
    got = eu.run_schedule(runner, prompts, steps, wants=wants)
    assert worst(got[0], want[0][n - 90:]) < F32_BOUND
    assert worst(got[1], want[1]) < F32_BOUND


# ------------------------------------------------------------------- long decoding
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding(dtype):
    cfg = ru.TINY_ALL
    model, tensors = build(cfg, seed=21, dtype=dtype)
    n = 330
    prompts = [ru.tokens(n, cfg["vocab"], 5)]
    want = plain_logits(cfg, tensors, prompts)[0]
    runner = runner_for(model, page_size=16, tokens=512)       # decode steps replay from graphs
    got = eu.run_schedule(runner, prompts, eu.bulk_then_single([n], tail=300))[0]
    if dtype == "float32":
        assert worst(got, want) < F32_BOUND
    else:
        assert_bfloat16_close(got, want)


# ------------------------------------------- unequal requests together and alone
def test_batch_against_each_alone():
    cfg = ru.TINY_ALL
    model, tensors = build(cfg, seed=2, dtype="bfloat16")
    lengths = [64, 3, 41, 17]
    prompts = [ru.tokens(n, cfg["vocab"], 40 + i) for i, n in enumerate(lengths)]
    alone = eu.run_schedule(runner_for(model, tokens=256), prompts, eu.whole(lengths))
    together = [([(i, 0, n) for i, n in enumerate(lengths)], list(range(len(lengths))))]
    got = eu.run_schedule(runner_for(model, tokens=256), prompts, together)
    assert_bfloat16_close(torch.cat(got), torch.cat(alone))


# ------------------------------------------- generation through engine and scheduler
def test_greedy_generation():
    from zig_ai_amd.engine import Engine
    cfg = ru.TINY_ALL
    d, tensors = ru.folder(cfg, seed=8)
    engine = Engine(d, dtype="float32", page_size=4, num_pages=128, max_num_seqs=3,
                    max_num_batched_tokens=48, chunk_size=20, max_model_len=256)
    prompts = [ru.tokens(n, cfg["vocab"], 60 + i) for i, n in enumerate([33, 5, 70, 12, 1])]
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
    cfg = ru.TINY_OTHER
    d, tensors = ru.folder(cfg, seed=8)
    engine = Engine(d, dtype="bfloat16", page_size=16, num_pages=64, max_num_seqs=4,
                    max_model_len=256)
    assert engine.runner.graphs is not None        # every part can be recorded
    prompts = [ru.tokens(n, cfg["vocab"], 80 + i) for i, n in enumerate([40, 7, 19])]
    outs = engine.generate(prompts, max_new_tokens=24, temperature=0.0)
    for p, o in zip(prompts, outs):
        logits = plain.forward(cfg, tensors, p + o)
        for j, tok in enumerate(o):
            row = logits[len(p) + j - 1]
            spread = float(row.max() - row.min())
            assert float(row.max() - row[tok]) <= 0.1 * spread, (j, tok)


# ------------------------------------------------------------------ kernels alone
def _slots(n_slots, floats, device):
    # rows spaced wider than their length, as the cache manager's slot rows are
    mem = torch.zeros((n_slots, floats + 12), dtype=torch.float32, device=device)
    return mem, mem[:, :floats]


def _step_arrays(lengths, slots, device):
    seq = [i for i, n in enumerate(lengths) for _ in range(n)]
    start = [0]
    for n in lengths:
        start.append(start[-1] + n)
    mk = lambda v: torch.tensor(v, dtype=torch.int32, device=device)
    return mk(seq), mk(start), mk(slots)


@pytest.mark.parametrize("taps,dtype", [(4, torch.float32), (2, torch.bfloat16), (1, torch.float32),
                                        (8, torch.bfloat16)])
def test_causal_conv_kernel(taps, dtype):
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(taps)
    C, col0, width = 70, 5, 90
    lengths_a, lengths_b = [13, 1, 2, 40], [1, 5, 1, 3]      # two steps of the same requests
    n_a, n_b = sum(lengths_a), sum(lengths_b)
    x = torch.randn(n_a + n_b, width, generator=g).to(dtype)
    w = torch.randn(C, taps, generator=g)
    bias = torch.randn(C, generator=g)
    mem, state = _slots(6, C * (taps - 1) + 7, dev)
    slots = [4, 0, 5, 2]
    xa, xb = x[:n_a].to(dev).contiguous(), x[n_a:].to(dev).contiguous()
    ya = ops.causal_conv_silu(xa, col0, w.to(dev), bias.to(dev), state, 7,
                              *_step_arrays(lengths_a, slots, dev)).cpu()
    yb = ops.causal_conv_silu(xb, col0, w.to(dev), bias.to(dev), state, 7,
                              *_step_arrays(lengths_b, slots, dev)).cpu()
    a0 = b0 = 0
    for la, lb in zip(lengths_a, lengths_b):
        whole = torch.cat([x[a0:a0 + la], x[n_a + b0:n_a + b0 + lb]]).double()[:, col0:col0 + C]
        want = plain.silu(plain.causal_conv(whole, w.double(), bias.double()))
        got = torch.cat([ya[a0:a0 + la], yb[b0:b0 + lb]]).double()
        assert float((got - want).abs().max()) < 1e-5
        a0, b0 = a0 + la, b0 + lb
    assert float(mem[:, C * (taps - 1) + 7:].abs().max()) == 0.0     # nothing beyond the window
    assert float(state[1].abs().max()) == 0.0                        # a slot nobody uses


def _plain_delta(q, k, v, beta, decay):
    T, H, d = decay.shape
    G, dv = q.shape[1], v.shape[2]
    out = torch.zeros((T, H, dv), dtype=torch.float64)
    for h in range(H):
        g = h // (H // G)
        S = torch.zeros((d, dv), dtype=torch.float64)
        for t in range(T):
            S = decay[t, h][:, None] * S
            u = beta[t, h] * (v[t, h] - S.T @ k[t, g])
            S = S + torch.outer(k[t, g], u)
            out[t, h] = S.T @ q[t, g]
    return out


@pytest.mark.parametrize("H,G,d,dv", [(2, 1, 16, 8), (3, 3, 40, 72), (2, 2, 128, 128), (4, 2, 64, 256),
                                      (1, 1, 256, 64)])
def test_delta_recurrence_kernel(H, G, d, dv):
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(d + dv)
    lengths = [37, 1, 18]
    T = sum(lengths)
    conv = torch.randn(T, 2 * G * d + H * dv + 3, generator=gen)
    proj = torch.randn(T, H + 5, generator=gen)
    decay_raw = torch.randn(T, H * d + 9, generator=gen)
    dt_bias = torch.randn(H * d, generator=gen)
    A_log = torch.rand(H, generator=gen) * 4 - 4
    mem, state = _slots(5, 11 + H * d * dv, dev)
    slots = [3, 0, 4]
    seq, start, slot_id = _step_arrays(lengths, slots, dev)
    # in two steps: the first tokens of every request, then the rest, through the state
    cut = [20, 0, 7]
    rows_a = [r for i, n in enumerate(lengths) for r in range(int(start[i]), int(start[i]) + cut[i])]
    rows_b = [r for i, n in enumerate(lengths) for r in range(int(start[i]) + cut[i], int(start[i + 1]))]
    got = torch.zeros((T, H * dv), dtype=torch.float64)
    for rows, lens, used in ((rows_a, [c for c in cut if c], [s for s, c in zip(slots, cut) if c]),
                             (rows_b, [n - c for n, c in zip(lengths, cut)], slots)):
        idx = torch.tensor(rows)
        _, st, sl = _step_arrays(lens, used, dev)
        out = ops.matrix_recurrence("delta", conv[idx].to(dev).contiguous(), 3, 3 + G * d,
                                    3 + 2 * G * d, proj[idx].to(dev).contiguous(), 5,
                                    decay_raw[idx].to(dev).contiguous(), dt_bias.to(dev),
                                    A_log.to(dev), None, state, 11, st, sl, H, G, d, dv)
        got[idx] = out.cpu().double()
    c = conv.double()
    for i in range(len(lengths)):
        a, b = int(start[i]), int(start[i + 1])
        q = c[a:b, 3:3 + G * d].view(-1, G, d)
        k = c[a:b, 3 + G * d:3 + 2 * G * d].view(-1, G, d)
        v = c[a:b, 3 + 2 * G * d:].view(-1, H, dv)
        q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
        k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        beta = torch.sigmoid(proj[a:b, 5:5 + H].double())
        decay = torch.exp(-torch.exp(A_log.double())[None, :, None] * plain.softplus(
            (decay_raw[a:b, :H * d].double() + dt_bias.double()).view(-1, H, d)))
        want = _plain_delta(q, k, v, beta, decay).reshape(b - a, H * dv)
        assert float((got[a:b] - want).abs().max()) < 2e-5 * max(1.0, float(want.abs().max()))
    assert float(mem[:, 11 + H * d * dv:].abs().max()) == 0.0
    assert float(state[:, :11].abs().max()) == 0.0


@pytest.mark.parametrize("H,G,N,P", [(4, 2, 24, 16), (3, 1, 128, 64), (2, 2, 16, 40)])
def test_ssd_recurrence_kernel(H, G, N, P):
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(N + P)
    lengths = [29, 2, 1]
    T = sum(lengths)
    conv = torch.randn(T, H * P + 2 * G * N, generator=gen)
    proj = torch.randn(T, 4 + H, generator=gen).to(torch.bfloat16)
    dt_bias, D = torch.randn(H, generator=gen), torch.randn(H, generator=gen)
    A_log = torch.rand(H, generator=gen) * 3 - 3
    mem, state = _slots(4, H * N * P, dev)
    seq, start, slot_id = _step_arrays(lengths, [2, 3, 0], dev)
    out = ops.matrix_recurrence("ssd", conv.to(dev), H * P + G * N, H * P, 0, proj.to(dev), 4, None,
                                dt_bias.to(dev), A_log.to(dev), D.to(dev), state, 0, start, slot_id,
                                H, G, N, P).cpu().double()
    c = conv.double()
    for i in range(len(lengths)):
        a, b = int(start[i]), int(start[i + 1])
        x = c[a:b, :H * P].view(-1, H, P)
        B = c[a:b, H * P:H * P + G * N].view(-1, G, N)
        C = c[a:b, H * P + G * N:].view(-1, G, N)
        dt = plain.softplus(proj[a:b, 4:].double() + dt_bias.double())
        for h in range(H):
            S = torch.zeros((N, P), dtype=torch.float64)
            for t in range(b - a):
                S = torch.exp(-torch.exp(A_log[h].double()) * dt[t, h]) * S \
                    + dt[t, h] * torch.outer(B[t, h // (H // G)], x[t, h])
                want = S.T @ C[t, h // (H // G)] + D[h].double() * x[t, h]
                assert float((out[a + t, h * P:(h + 1) * P] - want).abs().max()) < 2e-5 * max(
                    1.0, float(want.abs().max()))
    assert float(state[1].abs().max()) == 0.0


def _chunk_items(lengths, size, dev):
    seq, row0, cnt, r = [], [], [], 0
    for i, n in enumerate(lengths):
        for at in range(0, n, size):
            seq.append(i), row0.append(r + at), cnt.append(min(size, n - at))
        r += n
    return tuple(torch.tensor(v, dtype=torch.int32, device=dev) for v in (seq, row0, cnt)) + (len(seq),)


@pytest.mark.parametrize("H,G,d,dv,strong", [(2, 1, 16, 8, False), (3, 3, 40, 72, True), (2, 2, 128, 128, False),
                                             (4, 2, 64, 200, True), (1, 1, 31, 17, False), (2, 1, 64, 64, True),
                                             (2, 2, 32, 16, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_delta_recurrence_in_chunks(dtype, H, G, d, dv, strong):
    """Portions taken in chunks of 32 as matrix products: against float64, in two steps so that
    the second starts from carried states, with portions of exactly a chunk, one token more and
    fewer, half a chunk and one token; with decays down to zero; raw strengths and decays of either
    storage type; widths that fill the tiles of 32, 64 and 128 and ones that do not.  (Bound as for
    the walk.)"""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(d + dv)
    C = ops.DELTA_CHUNK
    steps = [[C + 1, 1, 2 * C, C - 1, 16], [C // 2 + 1, 70, 1, 5, C]]
    slots = [3, 0, 4, 5, 1]
    mem, state = _slots(7, 12 + H * d * dv, dev)
    A_log = torch.rand(H, generator=gen) * 4 - (1 if strong else 4)
    dt_bias = torch.randn(H * d, generator=gen)
    S64 = [torch.zeros(H, d, dv, dtype=torch.float64) for _ in slots]
    for lengths in steps:
        T = sum(lengths)
        conv = torch.randn(T, 2 * G * d + H * dv + 3, generator=gen)
        proj = torch.randn(T, H + 5, generator=gen).to(dtype)
        raw = (torch.randn(T, H * d + 9, generator=gen) * (8.0 if strong else 1.0)).to(dtype)
        _, start, slot_id = _step_arrays(lengths, slots, dev)
        out = ops.delta_recurrence_chunked(conv.to(dev), 3, 3 + G * d, 3 + 2 * G * d, proj.to(dev), 5, raw.to(dev),
                                           dt_bias.to(dev), A_log.to(dev), state, 12, slot_id,
                                           _chunk_items(lengths, C, dev), H, G, d, dv).cpu().double()
        c, r = conv.double(), 0
        for i, n in enumerate(lengths):
            rows = slice(r, r + n)
            q, k = c[rows, 3:3 + G * d].view(n, G, d), c[rows, 3 + G * d:3 + 2 * G * d].view(n, G, d)
            v = c[rows, 3 + 2 * G * d:].view(n, H, dv)
            q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5).repeat_interleave(H // G, 1)
            k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
            beta = torch.sigmoid(proj[rows, 5:5 + H].double())
            decay = torch.exp(-torch.exp(A_log.double())[None, :, None] * plain.softplus(
                (raw[rows, :H * d].double() + dt_bias.double()).view(n, H, d)))
            want = torch.zeros(n, H, dv, dtype=torch.float64)
            for t in range(n):
                S64[i] = decay[t][:, :, None] * S64[i]
                u = beta[t][:, None] * (v[t] - torch.einsum("hkv,hk->hv", S64[i], k[t]))
                S64[i] = S64[i] + k[t][:, :, None] * u[:, None, :]
                want[t] = torch.einsum("hkv,hk->hv", S64[i], q[t])
            assert float((out[rows] - want.reshape(n, -1)).abs().max()) < 2e-5 * max(1.0, float(want.abs().max()))
            r += n
        for i, slot in enumerate(slots):
            kept = state[slot, 12:].double().cpu().view(H, dv, d).transpose(1, 2)
            assert float((kept - S64[i]).abs().max()) < 2e-5 * max(1.0, float(S64[i].abs().max()))
    assert float(mem[:, 12 + H * d * dv:].abs().max()) == 0.0
    assert float(state[:, :12].abs().max()) == 0.0 and float(state[2].abs().max()) == 0.0


@pytest.mark.parametrize("H,G,N,P,strong", [(4, 2, 24, 16, True), (3, 1, 128, 64, False), (2, 2, 33, 130, False),
                                            (2, 1, 64, 128, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_ssd_recurrence_in_chunks(dtype, H, G, N, P, strong):
    """As above for a decay a head and token, in chunks of 128."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(N + P)
    C = ops.RETENTION_CHUNK
    steps = [[C + 1, 1, 2 * C + 16, C - 1], [40, C, 1, 17]]
    slots = [2, 3, 0, 4]
    mem, state = _slots(6, H * N * P, dev)
    dt_bias, D = torch.randn(H, generator=gen), torch.randn(H, generator=gen)
    A_log = torch.rand(H, generator=gen) * 3 - (0 if strong else 3)
    S64 = [torch.zeros(H, N, P, dtype=torch.float64) for _ in slots]
    for lengths in steps:
        T = sum(lengths)
        conv = torch.randn(T, H * P + 2 * G * N, generator=gen)
        proj = (torch.randn(T, 4 + H, generator=gen) * (6.0 if strong else 1.0)).to(dtype)
        _, start, slot_id = _step_arrays(lengths, slots, dev)
        out = ops.ssd_recurrence_chunked(conv.to(dev), H * P + G * N, H * P, 0, proj.to(dev), 4, dt_bias.to(dev),
                                         A_log.to(dev), D.to(dev), state, 0, slot_id,
                                         _chunk_items(lengths, C, dev), H, G, N, P).cpu().double()
        c, r = conv.double(), 0
        for i, n in enumerate(lengths):
            rows = slice(r, r + n)
            x = c[rows, :H * P].view(n, H, P)
            B = c[rows, H * P:H * P + G * N].view(n, G, N).repeat_interleave(H // G, 1)
            Cq = c[rows, H * P + G * N:].view(n, G, N).repeat_interleave(H // G, 1)
            dt = plain.softplus(proj[rows, 4:].double() + dt_bias.double())
            decay = torch.exp(-torch.exp(A_log.double()) * dt)
            want = torch.zeros(n, H, P, dtype=torch.float64)
            for t in range(n):
                S64[i] = decay[t][:, None, None] * S64[i] + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None, :]
                want[t] = torch.einsum("hnp,hn->hp", S64[i], Cq[t]) + D.double()[:, None] * x[t]
            assert float((out[rows] - want.reshape(n, -1)).abs().max()) < 2e-5 * max(1.0, float(want.abs().max()))
            r += n
        for i, slot in enumerate(slots):
            kept = state[slot].double().cpu().view(H, P, N).transpose(1, 2)
            assert float((kept - S64[i]).abs().max()) < 2e-5 * max(1.0, float(S64[i].abs().max()))
    assert float(mem[:, H * N * P:].abs().max()) == 0.0 and float(state[1].abs().max()) == 0.0


@pytest.mark.parametrize("H,G,N,P", [(8, 1, 128, 64), (3, 3, 64, 128), (2, 2, 128, 192), (64, 1, 64, 64)])
def test_ssd_chunks_off_their_boundaries(H, G, N, P):
    """Whole tiles, whose rows are read 16 bytes at a time, against the same rows a float further on, which
    are read one element at a time: the same bits, in chunks of one to a hundred and twenty-eight tokens."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(H + N + P)
    C = ops.RETENTION_CHUNK
    lengths, slots = [C + 1, 1, 2 * C + 16, C - 1, 17], [2, 3, 0, 4, 1]
    T, width = sum(lengths), H * P + 2 * G * N
    rand = lambda *shape: torch.randn(*shape, device=dev, generator=gen)
    x, proj, bias, A_log, D, first = rand(T, width), rand(T, H), rand(H), rand(H) - 1.0, rand(H), rand(6, H * N * P)
    x[C + 40, 3], x[5, H * P - 1] = math.inf, math.nan
    slot_id = torch.tensor(slots, dtype=torch.int32, device=dev)
    got = []
    for off in (0, 1):
        conv = torch.cat([rand(T, off), x, rand(T, 4 - off)], dim=1).contiguous()
        state = first.clone()
        out = ops.ssd_recurrence_chunked(conv, off + H * P + G * N, off + H * P, off, proj, 0, bias, A_log, D, state, 0,
                                         slot_id, _chunk_items(lengths, C, dev), H, G, N, P)
        got.append((out, state))
    for a, b in zip(*got):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    assert bool(torch.isfinite(got[0][0][C + 1:C + 2]).all()) and bool(torch.isnan(got[0][0]).any())


@pytest.mark.parametrize("H,G,N,P", [(8, 1, 128, 64), (3, 3, 64, 128), (2, 2, 128, 192)])
def test_ssd_chunks_with_values_off_their_boundaries(H, G, N, P):
    """Values that start one, two and three floats off a multiple of four, keys and queries on it: the bits of the
    same values on it, which take the kernels of whole tiles as well."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(H + N + P)
    C = ops.RETENTION_CHUNK
    lengths, slots = [C + 1, 1, 2 * C + 16, C - 1, 17], [2, 3, 0, 4, 1]
    T, keys = sum(lengths), G * N
    rand = lambda *shape: torch.randn(*shape, device=dev, generator=gen)
    values, k, q = rand(T, H * P), rand(T, keys), rand(T, keys)
    proj, bias, A_log, D, first = rand(T, H), rand(H), rand(H) - 1.0, rand(H), rand(6, H * N * P)
    slot_id = torch.tensor(slots, dtype=torch.int32, device=dev)
    base = None
    for off in (0, 1, 2, 3):
        conv = torch.cat([k, q, rand(T, off), values, rand(T, 4 - off)], dim=1).contiguous()
        state = first.clone()
        out = ops.ssd_recurrence_chunked(conv, keys, 0, 2 * keys + off, proj, 0, bias, A_log, D, state, 0, slot_id,
                                         _chunk_items(lengths, C, dev), H, G, N, P)
        base = base or (out, state)
        assert torch.equal(out, base[0]) and torch.equal(state, base[1]), off


@pytest.mark.parametrize("H,G,N,P", [(8, 1, 128, 64), (8, 2, 64, 128), (12, 3, 24, 16), (4, 1, 33, 130), (5, 1, 128, 70)])
def test_ssd_chunks_with_scores_worked_out_once(H, G, N, P, monkeypatch):
    """Heads that share keys and queries take their scores from one place: the bits of the same heads with
    keys and queries of their own, in chunks of one to a hundred and twenty-eight tokens (states of few
    rows too, which only many heads take this way by themselves)."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(H + N)
    C = ops.RETENTION_CHUNK
    lengths, slots = [C + 1, 1, 2 * C + 16, C - 1, 17], [2, 3, 0, 4, 1]
    T, per = sum(lengths), H // G
    assert ops.shares_scores(64, 64 // per, N) and not ops.shares_scores(H, H, N)
    monkeypatch.setattr(ops, "shares_scores", lambda heads, groups, dk: heads > groups)
    x, B, Q = (torch.randn(T, n, generator=gen) for n in (H * P, G * N, G * N))
    proj = torch.randn(T, H, generator=gen)
    dt_bias, D, A_log = (torch.randn(H, generator=gen).to(dev) for _ in range(3))
    _, start, slot_id = _step_arrays(lengths, slots, dev)
    results = []
    for groups, q, k in ((G, Q, B), (H, *(y.view(T, G, N).repeat_interleave(per, 1).reshape(T, H * N) for y in (Q, B)))):
        _, state = _slots(6, H * N * P, dev)
        conv = torch.cat([x, k, q], dim=1).to(dev)
        out = ops.ssd_recurrence_chunked(conv, H * P + groups * N, H * P, 0, proj.to(dev), 0, dt_bias, A_log, D, state, 0,
                                         slot_id, _chunk_items(lengths, C, dev), H, groups, N, P)
        results.append((out, state.clone()))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("strength", [1e3, 1e5, 1e7, 1e30])
def test_ssd_chunks_behind_a_token_that_forgets(strength):
    """A few tokens whose decay is zero (``exp(A_log) dt`` = ``strength``) among tokens that keep
    three quarters: what the former leave decays at the latter's pace.  (Bound as above.)"""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(7)
    H, G, N, P, C = 2, 1, 32, 48, ops.RETENTION_CHUNK
    lengths, slots = [C + 70, 33], [1, 0]
    T = sum(lengths)
    mem, state = _slots(2, H * N * P, dev)
    conv = torch.randn(T, H * P + 2 * G * N, generator=gen)
    proj = math.log(0.3 / (strength / 5)) + 0.1 * torch.randn(T, H, generator=gen)
    for t in (0, 17, 60, 61, 100, C + 3, C + 90):
        proj[t, 0], proj[min(t + 1, T - 1), 1] = 5.0, 5.0
    A_log, bias = torch.full((H,), math.log(strength / 5)), torch.zeros(H)
    _, start, slot_id = _step_arrays(lengths, slots, dev)
    out = ops.ssd_recurrence_chunked(conv.to(dev), H * P + G * N, H * P, 0, proj.to(dev), 0, bias.to(dev),
                                     A_log.to(dev), bias.to(dev), state, 0, slot_id,
                                     _chunk_items(lengths, C, dev), H, G, N, P).cpu().double()
    c, dt = conv.double(), plain.softplus(proj.double())
    decay = torch.exp(-torch.exp(A_log.double()) * dt)
    for i, slot in enumerate(slots):
        S = torch.zeros(H, N, P, dtype=torch.float64)
        for t in range(int(start[i]), int(start[i + 1])):
            S = decay[t][:, None, None] * S + torch.outer(dt[t], c[t, H * P:H * P + N])[:, :, None] \
                * c[t, :H * P].view(H, 1, P)
            want = torch.einsum("hnp,n->hp", S, c[t, H * P + N:]).reshape(-1)
            assert float((out[t] - want).abs().max()) < 2e-5 * max(1.0, float(want.abs().max())), t
        kept = state[slot].double().cpu().view(H, P, N).transpose(1, 2)
        assert float((kept - S).abs().max()) < 2e-5 * max(1.0, float(S.abs().max()))


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("at", [5, 20, 64, 127, 130])
def test_ssd_chunks_keep_a_bad_value_from_earlier_tokens(bad, at):
    """A token's value that is infinite or not a number stays in its column, from its token on."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(at)
    H, G, N, P, C = 2, 1, 40, 72, ops.RETENTION_CHUNK
    lengths, slots = [7, C + 20, 9], [1, 0, 2]
    T, first = sum(lengths), lengths[0]
    conv = torch.randn(T, H * P + 2 * G * N, generator=gen).to(dev)
    proj = torch.randn(T, H, generator=gen).to(dev)
    A_log, bias = torch.full((H,), -2.0, device=dev), torch.zeros(H, device=dev)
    _, _, slot_id = _step_arrays(lengths, slots, dev)

    def run(x):
        _, state = _slots(3, H * N * P, dev)
        out = ops.ssd_recurrence_chunked(x, H * P + G * N, H * P, 0, proj, 0, bias, A_log, bias, state, 0, slot_id,
                                         _chunk_items(lengths, C, dev), H, G, N, P)
        return out.view(T, H, P)

    want = run(conv)
    spoilt = conv.clone()
    spoilt[first + at, 70] = bad                     # head 0, column 70
    got = run(spoilt)
    after = torch.zeros(T, H, P, dtype=torch.bool, device=dev)
    after[first + at:first + lengths[1], 0, 70] = True
    assert bool((~torch.isfinite(got[after])).all())
    assert float((got - want)[~after].abs().max()) < 2e-5 * float(want.abs().max())


@pytest.mark.parametrize("d,dv", [(128, 128), (40, 24), (16, 16)])
@pytest.mark.parametrize("last", [1, 17, 32])
@pytest.mark.parametrize("chunks", [3, 4, 5, 6, 7])
def test_delta_chunks_far_ahead(chunks, last, d, dv):
    """A portion of several chunks, walked with the next ones' operands on their way, leaves the bits
    that its chunks leave one call after the other (the state between them is 32-bit either way)."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(chunks)
    H, C = 2, ops.DELTA_CHUNK
    T = (chunks - 1) * C + last
    conv = torch.randn(T, 2 * H * d + H * dv, generator=gen).to(dev)
    proj, raw = torch.randn(T, H, generator=gen).to(dev), torch.randn(T, H * d, generator=gen).to(dev)
    A_log, bias = torch.full((H,), -2.0, device=dev), torch.zeros(H * d, device=dev)
    start = torch.randn(H * d * dv, generator=gen).to(dev)

    def run(portions):
        _, state = _slots(2, H * d * dv, dev)
        state[1] = start
        out, at = [], 0
        for n in portions:
            rows = slice(at, at + n)
            out.append(ops.delta_recurrence_chunked(
                conv[rows], 0, H * d, 2 * H * d, proj[rows], 0, raw[rows], bias, A_log, state, 0,
                torch.tensor([1], dtype=torch.int32, device=dev), _chunk_items([n], C, dev), H, H, d, dv))
            at += n
        return torch.cat(out), state

    (whole, state), (parts, want) = run([T]), run([C] * (chunks - 1) + [last])
    assert torch.equal(whole, parts) and torch.equal(state, want)


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("at", [5, 16, 20, 31, 40, 69])
def test_delta_chunks_keep_a_bad_value_from_earlier_tokens(bad, at):
    """The same for the delta rule, and for a key and a write strength (which spoil their head)."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(at)
    H, G, d, dv = 2, 2, 40, 24
    lengths, slots = [7, 70, 9], [1, 0, 2]
    T, first = sum(lengths), lengths[0]
    conv = torch.randn(T, 2 * G * d + H * dv, generator=gen).to(dev)
    proj = torch.randn(T, H, generator=gen).to(dev)
    raw = torch.randn(T, H * d, generator=gen).to(dev)
    A_log, bias = torch.full((H,), -2.0, device=dev), torch.zeros(H * d, device=dev)
    _, _, slot_id = _step_arrays(lengths, slots, dev)

    def run(x, strength):
        _, state = _slots(3, H * d * dv, dev)
        out = ops.delta_recurrence_chunked(x, 0, G * d, 2 * G * d, strength, 0, raw, bias, A_log, state, 0, slot_id,
                                           _chunk_items(lengths, ops.DELTA_CHUNK, dev), H, G, d, dv)
        return out.view(T, H, dv)

    want = run(conv, proj)
    value, key, strength = conv.clone(), conv.clone(), proj.clone()
    value[first + at, 2 * G * d + 17] = bad          # head 0, column 17
    key[first + at, G * d + 3] = bad
    strength[first + at, 0] = math.nan
    rows = slice(first + at, first + lengths[1])
    for got, columns in ((run(value, proj), slice(17, 18)), (run(key, proj), slice(0, dv)),
                         (run(conv, strength), slice(0, dv))):
        after = torch.zeros(T, H, dv, dtype=torch.bool, device=dev)
        after[rows, 0, columns] = True
        assert bool((~torch.isfinite(got[after])).all())
        assert float((got - want)[~after].abs().max()) < 2e-5 * float(want.abs().max())


@pytest.mark.parametrize("kind", ["ssd", "delta", "delta wide"])
def test_a_portion_takes_its_form_by_its_own_length(kind):
    """Single tokens and short portions of a request give the same bits alone and beside a portion
    that is taken in chunks, which gives the same bits alone and beside them (32-bit, where every
    other part sums in an order of its own too)."""
    from zig_ai_amd.kernels import ops
    cfg = ALONE[kind]
    model, _ = build(cfg, seed=5)
    n = ops.CHUNKED_FROM
    prompts = [ru.tokens(14, cfg["vocab"], 1), ru.tokens(2 * n + 40, cfg["vocab"], 2)]
    short = [(0, 0, 3), (0, 3, 4), (0, 4, 5), (0, 5, 13), (0, 13, 14)]
    long = [(1, 0, n), (1, n, n + 40), (1, n + 40, 2 * n + 40)]

    def run(schedule):
        return eu.run_schedule(runner_for(model, tokens=2 * n + 80), prompts, schedule)

    alone = run([([e], []) for e in short[:-1]] + [([short[-1]], [0])] + [([e], []) for e in long[:-1]]
                + [([long[-1]], [1])])
    beside = run([([short[0]], []), ([short[1], long[0]], []), ([long[1], short[2]], []),
                  ([short[3], long[2]], [1]), ([short[4]], [0])])
    for a, b in zip(alone, beside):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["ssd", "delta"])
def test_recorded_steps_with_both_forms(kind):
    """A step of one token beside a portion in chunks, recorded and replayed with other requests: the
    bits of the same steps run as they are."""
    from zig_ai_amd.engine import ModelRunner
    from zig_ai_amd.kernels import ops
    cfg = ALONE[kind]
    model, _ = build(cfg, seed=6)
    n, rounds = ops.CHUNKED_FROM + 5, 5
    prompts = [ru.tokens(3 + rounds, cfg["vocab"], 1)] + [ru.tokens(n, cfg["vocab"], 2 + i) for i in range(rounds)]
    schedule = [([(0, 0, 3)], [])] + [([(0, 3 + i, 4 + i), (1 + i, 0, n)], [1 + i] + ([0] if i == rounds - 1 else []))
                                      for i in range(rounds)]
    recorded, plain_run = (ModelRunner(model, page_size=4, num_pages=n, num_slots=3, use_graphs=graphs,
                                       portion_graphs=graphs) for graphs in (True, False))
    got, want = (eu.run_schedule(r, prompts, schedule) for r in (recorded, plain_run))
    assert recorded.graphs.portion_replays >= rounds - 2
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("form", ["ssd", "delta", "fixed"])
def test_the_walk_of_short_portions_alone(form):
    """With a limit the walk takes the shorter portions, to the bit as in a step of their own, and
    leaves the others' rows and states alone."""
    from zig_ai_amd.engine.batch import ShortPortions
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(3)
    H, G, d, dv, limit = 4, 2 if form != "fixed" else 4, 24, 40, 192
    lengths, slots = [3, limit, 1, limit - 1, 250, 17], [3, 0, 5, 1, 6, 2]
    conv = torch.randn(sum(lengths), 2 * G * d + H * dv, generator=gen).to(dev)
    proj = torch.randn(sum(lengths), H, generator=gen).to(dev)
    raw = torch.randn(sum(lengths), H * d, generator=gen).to(dev)
    heads, channels = torch.rand(H, generator=gen).to(dev), torch.randn(H * d, generator=gen).to(dev)
    before = torch.randn(7, H * d * dv, generator=gen).to(dev)

    def walk(rows, lens, used, state, **kw):
        _, start, slot_id = _step_arrays(lens, used, dev)
        return ops.matrix_recurrence(
            form, conv[rows].contiguous(), 0, G * d, 2 * G * d, None if form == "fixed" else proj[rows].contiguous(),
            0, {"ssd": None, "fixed": heads}.get(form, raw[rows].contiguous()),
            channels if form == "delta" else heads, heads, heads, state, 0, start, slot_id, H, G, d, dv, **kw)

    short = [i for i, n in enumerate(lengths) if n < limit]
    rows_of = [slice(sum(lengths[:i]), sum(lengths[:i + 1])) for i in range(len(lengths))]
    lens = [lengths[i] for i in short]
    out = torch.full((sum(lengths), H * dv), 7.0, device=dev)
    state = before.clone()
    walk(slice(None), lengths, slots, state, short=ShortPortions(limit, len(lens), sum(lens), max(lens)), out=out)
    alone = before.clone()
    idx = torch.cat([torch.arange(rows_of[i].start, rows_of[i].stop) for i in short]).to(dev)
    want = walk(idx, lens, [slots[i] for i in short], alone)
    assert torch.equal(out[idx], want) and torch.equal(state, alone)
    for i in range(len(lengths)):
        if i not in short:
            assert bool((out[rows_of[i]] == 7.0).all()) and torch.equal(state[slots[i]], before[slots[i]])


def test_small_kernels():
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(0)
    T = 9
    for I in (52, 56):          # element by element, and eight at a time
        gu = (torch.randn(T, 2 * I, generator=gen) * 3).to(torch.bfloat16)
        got = ops.clamped_glu(gu.to(dev), 2.0, 1.702, 1.0).cpu().double()
        g = gu[:, :I].double().clamp(max=2.0)
        u = gu[:, I:].double().clamp(-2.0, 2.0)
        want = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        assert float((got - want).abs().max()) < 0.04
        got = ops.clamped_glu(gu.float().to(dev), 2.0, 1.702, 1.0).cpu().double()
        assert float((got - want).abs().max()) < 1e-5
    # gated group norm, both orders
    y = torch.randn(T, 96, generator=gen)
    gate = torch.randn(T, 96 + 8, generator=gen)
    w = torch.randn(96, generator=gen)
    got = ops.gated_group_norm(y.to(dev), gate.to(dev), 8, w.to(dev), 32, 1e-5, "silu", True).cpu()
    v = (y.double() * plain.silu(gate[:, 8:].double())).view(T, 3, 32)
    want = (plain.rms(v, 1e-5).reshape(T, 96) * w.double())
    assert float((got.double() - want).abs().max()) < 1e-5
    got = ops.gated_group_norm(y.to(dev), gate.to(dev), 8, w[:24].contiguous().to(dev), 24, 1e-5,
                               "sigmoid", False).cpu()
    want = (plain.rms(y.double().view(T, 4, 24), 1e-5) * w[:24].double()).reshape(T, 96) \
        * torch.sigmoid(gate[:, 8:].double())
    assert float((got.double() - want).abs().max()) < 1e-5
    # weighted additions to the stream, with and without the norm
    x = torch.randn(T, 80, generator=gen)
    a, b = torch.randn(T, 80, generator=gen), torch.randn(T, 80, generator=gen)
    nw = torch.randn(80, generator=gen)
    res = x.to(dev).clone()
    out = ops.scaled_add_rmsnorm(res, a.to(dev), 0.3, b.to(dev), -1.1, nw.to(dev), 1e-6).cpu()
    s = x.double() + 0.3 * a.double() - 1.1 * b.double()
    assert float((res.cpu().double() - s).abs().max()) < 1e-5
    assert float((out.double() - plain.rms(s, 1e-6) * nw.double()).abs().max()) < 1e-5
    assert ops.scaled_add_rmsnorm(res, a.to(torch.bfloat16).to(dev), 2.0) is None
    s = s + 2.0 * a.to(torch.bfloat16).double()
    assert float((res.cpu().double() - s).abs().max()) < 1e-5


@pytest.mark.parametrize("width", [4, 252, 1020, 1024, 1028, 2052, 3076, 4096, 4100, 33])
def test_rows_in_registers_at_the_edges_of_a_workgroup(width):
    """The three norms that keep a row in registers, at rows that do and do not fill a
    workgroup's vectors, and rows beyond them; a stack of partial sums with every count."""
    from zig_ai_amd.kernels import ops
    dev, T = torch.device("cuda"), 3
    g = torch.Generator().manual_seed(width)
    x, a, b = (torch.randn(T, width, generator=g) for _ in range(3))
    w = torch.randn(width, generator=g)
    res = x.to(dev).clone()
    out = ops.scaled_add_rmsnorm(res, a.to(dev), 0.3, b.to(dev), -1.1, w.to(dev), 1e-6)
    s = x.double() + 0.3 * a.double() - 1.1 * b.double()
    assert float((res.cpu().double() - s).abs().max()) < 1e-5
    assert float((out.cpu().double() - plain.rms(s, 1e-6) * w.double()).abs().max()) < 2e-5
    # (up to nine 32-bit additions before the norm, which for four elements may divide by little)
    for n in (1, 2, 8, 9):
        y = torch.randn(n, T, width, generator=g)
        res = x.to(dev).clone()
        out = ops.add_rmsnorm(res, y.to(dev), w.to(dev), 1e-6, torch.float32)
        s = x.double() + y.double().sum(0)
        assert float((res.cpu().double() - s).abs().max()) < 2e-5
        assert float((out.cpu().double() - plain.rms(s, 1e-6) * w.double()).abs().max()) < 4e-5
        res = x.to(dev).clone()
        ops.normed_add_(res, y.to(dev), w.to(dev), 1e-6, 0.5)
        s = x.double() + 0.5 * plain.rms(y.double().sum(0), 1e-6) * w.double()
        assert float((res.cpu().double() - s).abs().max()) < 4e-5


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
def test_causal_conv_at_the_edges_of_its_blocks(taps):
    """Portions that end before, on and behind a block of 16 tokens, shorter than the taps and of
    one token; 300 channels behind eight others."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(taps)
    lengths, slots, C, col0 = [15, 1, 17, 2, 32, 3, 16], [6, 0, 3, 1, 7, 2, 5], 300, 8
    x = torch.randn(sum(lengths), C + col0 + 4, generator=g).to(torch.bfloat16)
    w, b = torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    _, state = _slots(8, C * (taps - 1) + 4, dev)
    # (twice: the second time behind the first)
    got = [ops.causal_conv_silu(x.to(dev), col0, w.to(dev), b.to(dev), state, 4,
                                *_step_arrays(lengths, slots, dev)).cpu().double() for _ in range(2)]
    at = 0
    for n in lengths:
        rows = x[at:at + n, col0:col0 + C].double()
        want = plain.silu(plain.causal_conv(torch.cat([rows, rows]), w.double(), b.double()))
        assert float((torch.cat([y[at:at + n] for y in got]) - want).abs().max()) < 1e-5
        at += n


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,width,group,weights", [
    (1, 32, 32, 32), (3, 96, 32, 96), (67, 320, 64, 1), (5, 512, 256, 256), (9, 768, 96, 768), (130, 260, 260, 260),
    (2, 3072, 1024, 3072), (7, 1028, 1028, 1028), (3, 4096, 2048, 2048), (2, 4096, 4096, 4096), (2, 4100, 4100, 4100),
    (4, 600, 300, 1)])
def test_gated_group_norm_forms(dtype, T, width, group, weights):
    """Groups within a wave, a workgroup's, and those that go column by column (widths that are no power of two,
    one weight for wide groups), each with the gate before and behind the norm, on and off its boundaries."""
    from zig_ai_amd.kernels import ops
    dev = torch.device("cuda")
    gen = torch.Generator().manual_seed(width + group)
    y, w = torch.randn(T, width, generator=gen), torch.randn(weights, generator=gen)
    for off in (8, 3):
        gate = torch.randn(T, width + off, generator=gen).to(dtype)
        g, wide = gate[:, off:].double(), w.double().repeat(width // weights)
        for first, act in ((True, "silu"), (False, "sigmoid")):
            a = plain.silu(g) if act == "silu" else torch.sigmoid(g)
            v = y.double() * a if first else y.double()
            want = plain.rms(v.view(T, -1, group), 1e-5).reshape(T, width) * wide * (1.0 if first else a) * 0.75
            got = ops.gated_group_norm(y.to(dev), gate.to(dev), off, w.to(dev), group, 1e-5, act, first, 0.75)
            assert got.dtype == dtype
            # (32-bit sums of up to 4,100 squares; the one rounding to bfloat16 is 2^-9 of a value)
            tol = 1e-5 if dtype == torch.float32 else 2.0 ** -8
            assert float(((got.cpu().double() - want).abs() / want.abs().clamp(min=1.0)).max()) < tol, (off, first)
