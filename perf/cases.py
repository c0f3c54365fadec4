"""The work the engine's speed is measured on: steps of ``ModelRunner``, the one way in that
generation, trace replay and the benchmark all take, at the sizes ``bench.py`` runs and at
generic ones around them, for every design the engine serves.

A case is a step, or the few steps of a prompt that is cut into portions:

    design, width, dtype         the model: layer sizes as bench.py has them
    decoding, context, ragged    requests that bring one token each, and their longest context
                                 (all of that length, or spread from a quarter of it)
    prompts, prompt, portion     prompts that start in this step, the longest one's length, and
                                 the most tokens of one that a step takes (0: all)
    reproducible                 every sum in a fixed order

``draw`` takes every design through all of that: single requests and batches, short and long,
both directions, both storage types.

The weights are random.  Routers are the exception: a token's embedding carries one of sixteen
directions and a router's rows point along them, with a wide gap between the experts a token
takes and the rest, as a trained router's choices have; which expert runs then does not hang on
a last place, and outputs can be compared.
"""

import math
import random
import zlib

import torch

from zig_ai_amd.config import config_from_dict
from zig_ai_amd.engine import DecoderModel, ModelRunner, StepEntry
from zig_ai_amd.parts import Runtime
from zig_ai_amd.weights.loader import expected_tensors, keep_dtype

VOCAB, PAGE, CLASSES = 65536, 16, 16
WARM = 3                    # decode steps before a state is handed over (a recording is made at the second)
DT = torch.float64


# ------------------------------------------------------------------------ designs
def lfm2(hidden, heads, ff, layers, attention_at):
    return {"architectures": ["Lfm2ForCausalLM"], "model_type": "lfm2", "hidden_size": hidden,
            "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": 8,
            "vocab_size": VOCAB, "block_ff_dim": ff, "block_auto_adjust_ff_dim": True,
            "block_multiple_of": 256, "block_ffn_dim_multiplier": 1.0, "rope_theta": 1000000.0,
            "norm_eps": 1e-5, "conv_L_cache": 3, "conv_bias": False, "tie_embedding": True,
            "max_position_embeddings": 128000,
            "layer_types": ["full_attention" if i in attention_at else "conv" for i in range(layers)]}


def other(name, layers, eps, **more):
    return dict({"architecture": name, "vocab": VOCAB, "norm": {"eps": eps}, "layers": layers,
                 "max_position_embeddings": 128000}, **more)


def spread_decays(heads):
    return [1.0 - 2.0 ** -(5 + 7 * h / max(1, heads - 1)) for h in range(heads)]


def rudilix(width):
    heads = width // 128
    attention = {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128,
                 "scale": 128 ** -0.5, "mask": {"size": 1024}, "rot": {"dims": 64, "base": 1e6}}
    delta = {"heads": heads, "kv_heads": heads, "dim": 128, "vdim": 128, "conv": 4,
             "decay_rank": 64, "gate_rank": 64}
    ssd = {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 1, "norm_groups": 1, "conv": 4}
    both = {"left": attention, "right": dict(delta, heads=heads // 2, kv_heads=heads // 2),
            "left_scale": 1.0, "right_scale": 1.0}
    kinds = [("parallel", both), ("mamba2", ssd), ("channel_delta", delta), ("mamba2", ssd)]
    mlp = {"kind": "dense", "ff": 4 * width, "limit": 7.0}
    return other("Rudilix", [{"type": kinds[i % 4][0], "mixer": kinds[i % 4][1], "mlp": mlp}
                             for i in range(8)], 1e-5, width=width, residual_mult=1.0)


def ranesun(width):
    heads, q_heads = width // 128, width // 64
    kinds = [("retention", {"heads": heads, "dim": 64, "vdim": 128, "decay": spread_decays(heads),
                            "rot": {"dims": 64, "base": 5e5}}),
             ("attention", {"heads": q_heads, "kv_heads": max(1, q_heads // 8), "dim": 64, "vdim": 64,
                            "scale": 0.125, "softcap": 50.0, "q_temp": {"coef": 0.25, "every": 1024}})]
    mlps = [{"kind": "dense", "ff": 4 * width},
            {"kind": "moe", "expert": {"ff": 2 * width}, "router": {"experts": 8, "top": 2}}]
    return other("Ranesun", [{"type": kinds[i % 2][0], "mixer": kinds[i % 2][1], "mlp": mlps[i // 2 % 2]}
                             for i in range(8)], 1e-5, width=width, logit_scale=1.0,
                 loop={"start": 0, "stop": 4, "times": 1})


def gemodra(width):
    rotated = {"heads": width // 128, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512,
               "q_rank": 3 * width // 4, "scale": 192 ** -0.5, "rot": {"dims": 64, "base": 1e6}}
    plain = {k: v for k, v in dict(rotated, scale=128 ** -0.5).items() if k not in ("rot_dim", "rot")}
    mlp = {"kind": "moe", "expert": {"ff": width // 2}, "shared": {"ff": width},
           "router": {"experts": 30, "identity": 2, "top": 4, "scale": 2.0,
                      "groups": {"count": 4, "keep": 2}}}
    return other("Gemodra", [{"type": "latent_attention" + ("_2" if i % 4 == 3 else ""),
                              "mixer": plain if i % 4 == 3 else rotated, "mlp": mlp} for i in range(8)],
                 1e-6, width=width, residual_mult=0.5, logit_softcap=30.0, token_side={"dim": 256})


def nopozen(width):
    heads, q_heads = width // 128, width // 64
    lightning = {"heads": heads, "dim": 128, "vdim": 128, "decay": spread_decays(heads)}
    kinds = [("lightning", lightning),
             ("attention_2", {"heads": q_heads, "kv_heads": max(1, q_heads // 8), "dim": 64, "vdim": 64,
                              "scale": 0.125, "conv": 4, "rot": {"dims": 32, "base": 1e6}}),
             ("lightning", lightning),
             ("attention", {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128,
                            "scale": 128 ** -0.5, "mask": {"size": 1024},
                            "rot": {"dims": 128, "base": 5e5,
                                    "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}})]
    mlps = [{"kind": "dense", "ff": 4 * width},
            {"kind": "moe", "expert": {"ff": 2 * width}, "router": {"experts": 8, "top": 2}}]
    return other("Nopozen", [{"type": kinds[i % 4][0], "mixer": kinds[i % 4][1], "mlp": mlps[i // 2 % 2]}
                             for i in range(8)], 1e-6, width=width, loop={"start": 0, "stop": 4, "times": 1})


def vupelorn(width):
    linear = {"heads": width // 128, "dim": 128, "vdim": 128, "tau": 16.0, "decay_rank": 16}
    latent = {"heads": width // 128, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512,
              "q_rank": 3 * width // 4, "scale": 192 ** -0.5, "rot": {"dims": 64, "base": 1e6}}
    stretched = dict(latent, rot=dict(latent["rot"], scaling={"factor": 8.0, "original": 4096,
                                                              "fast": 32.0, "slow": 1.0}))
    mlp = {"kind": "moe", "expert": {"ff": width // 2, "limit": 7.0}, "router": {"experts": 32, "top": 4}}
    kinds = [("gla", linear), ("latent_attention_2", latent), ("gla", linear), ("latent_attention", stretched),
             ("gla", linear), ("latent_attention_2", dict(latent, kv_from=1)), ("gla", linear),
             ("latent_attention", stretched)]
    return other("Vupelorn", [{"type": k, "mixer": m, "mlp": mlp} for k, m in kinds], 1e-6, width=width,
                 embedding={"bigram": {"buckets": VOCAB - 1, "mul_prev": 31337, "mul_cur": 17}})


def torisun(width):
    heads = width // 128
    own = {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 64, "scale": 128 ** -0.5,
           "mask": {"size": 1024, "keep_first": 4},
           "rot": {"dims": 128, "base": 5e5, "scaling": {"factor": 8.0, "original": 4096,
                                                         "fast": 32.0, "slow": 1.0}}}
    mlps = [{"kind": "dense", "ff": 4 * width, "limit": 7.0},
            {"kind": "moe", "expert": {"ff": width // 2}, "shared": {"ff": width // 2},
             "router": {"experts": 32, "top": 4, "scale": 2.5}}]
    return other("Torisun", [{"type": "attention", "mixer": own if i % 2 == 0 else dict(own, kv_from=i - 1),
                              "mlp": mlps[i % 2]} for i in range(8)], 1e-6, width=width)


LFM2 = {"lfm2-350m": lfm2(1024, 16, 6656, 16, (2, 5, 8, 10, 12, 14)),
        "lfm2-1.2b": lfm2(2048, 32, 12288, 16, (2, 5, 8, 10, 12, 14)),
        "lfm2-2.6b": lfm2(2048, 32, 10752, 30, (2, 6, 10, 14, 18, 21, 24, 27))}
OTHERS = {"rudilix": rudilix, "ranesun": ranesun, "gemodra": gemodra, "nopozen": nopozen,
          "vupelorn": vupelorn, "torisun": torisun}


def config_of(case):
    return LFM2[case["design"]] if case["design"] in LFM2 else OTHERS[case["design"]](case["width"])


# -------------------------------------------------------------------------- cases
def case_of(design, decoding=0, context=0, ragged=False, prompts=0, prompt=0, portion=0,
            dtype="bfloat16", width=2048, reproducible=False, name=None):
    out = {} if name is None else {"name": name}
    if design in LFM2:
        width = LFM2[design]["hidden_size"]
    return dict(out, design=design, width=width, dtype=dtype, decoding=decoding, context=context,
                ragged=ragged, prompts=prompts, prompt=prompt, portion=portion, reproducible=reproducible)


def listed():
    return [
        # one user's chat with the smallest model, early in it: what a token's latency is
        case_of("lfm2-350m", 1, 60, name="chat 350m b1"),
        # the headline: eight requests at 2,048 tokens
        case_of("lfm2-1.2b", 8, 2048, name="decode 1.2b b8"),
        # a full server, its requests at different places
        case_of("lfm2-1.2b", 64, 2000, ragged=True, name="decode 1.2b b64"),
        # a prompt of 2,048 tokens alone
        case_of("lfm2-1.2b", prompts=1, prompt=2048, name="prompt 1.2b 2048"),
        # a long document coming in by portions beside requests that decode
        case_of("lfm2-2.6b", 13, 1500, ragged=True, prompts=1, prompt=5000, portion=1024, name="mixed 2.6b"),
        # a few short questions in the 32-bit mode (checks against other implementations)
        case_of("lfm2-350m", prompts=3, prompt=150, ragged=True, dtype="float32", name="prompts 350m f32"),
        # the other designs, at the sizes the benchmark compares them at, in each direction
        case_of("rudilix", prompts=1, prompt=2048, name="prompt rudilix"),
        case_of("ranesun", prompts=6, prompt=500, ragged=True, name="prompts ranesun"),
        case_of("gemodra", 8, 2048, name="decode gemodra b8"),
        case_of("nopozen", 20, 900, ragged=True, name="decode nopozen b20"),
        case_of("vupelorn", prompts=1, prompt=1777, name="prompt vupelorn"),
        case_of("torisun", 5, 1200, ragged=True, prompts=2, prompt=1000, portion=512, name="mixed torisun"),
    ]


def draw(rng):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    # LFM2 is what most of the work is; the others share the rest
    design = rng.choice(sorted(LFM2)) if rng.random() < 0.4 else rng.choice(sorted(OTHERS))
    width = rng.choice([1024, 2048])
    exact_32 = rng.random() < 0.12
    dtype = "float32" if exact_32 else "bfloat16"
    kind = rng.choice(["decode", "prompts", "mixed"])
    reproducible = rng.random() < 0.12
    most = 512 if exact_32 else 4096
    decoding = context = prompts = prompt = portion = 0
    if kind != "prompts":
        decoding = spread(1, 64 if kind == "decode" else 32)
        context = spread(16, min(4096, 80000 // decoding))
    if kind != "decode":
        prompts = spread(1, 8)
        prompt = spread(4, most // prompts)
    if kind == "mixed":
        portion = rng.choice([256, 512, 1024])
    return case_of(design, decoding, context, rng.random() < 0.7, prompts, prompt, portion, dtype, width,
                   reproducible)


# ------------------------------------------------------------------------- inputs
def token_class(tokens):
    """The direction (0 to CLASSES - 1) in a token's embedding; some are more frequent than others."""
    u = ((tokens.to(torch.int64) * 40503) % 65536).to(torch.float32) / 65536
    return (CLASSES * u ** 1.4).to(torch.int64)


def directions(width, device):
    """CLASSES orthogonal rows of signs."""
    i = torch.arange(width, device=device)
    rows = []
    for c in range(1, CLASSES + 1):
        bits, parity = i & c, torch.zeros_like(i)
        while int(bits.max()):
            parity, bits = parity ^ (bits & 1), bits >> 1
        rows.append(1.0 - 2.0 * parity.to(torch.float32))
    return torch.stack(rows)


def taken_experts(name, router, c):
    """The experts that tokens of one class take (as many as the router keeps, from two of its
    groups where it has groups)."""
    rng = random.Random(f"{name} {c}")
    n, top = int(router["experts"]) + int(router.get("identity", 0)), int(router["top"])
    groups = router.get("groups")
    if not groups:
        return rng.sample(range(n), top)
    per = n // int(groups["count"])
    kept = rng.sample(range(int(groups["count"])), int(groups["keep"]))
    share = -(-top // len(kept))
    return [g * per + e for g in kept for e in rng.sample(range(per), share)][:top]


# where a tensor's values lie by the end of its name: (mean, deviation); the first that fits
# (per design: what a name's end means can differ)
# (what a sublayer adds is small beside the stream, as trained models have it: rounding then
# does not grow from layer to layer)
VALUES = {
    "Lfm2": [("embed_tokens.weight", 0.0, 0.3), ("out_proj.weight", 0.0, 0.005), ("w2.weight", 0.0, 0.005)],
    "Rudilix": [("embed", 0.0, 0.5), ("mix.norm", 1.0, 0.1), ("right.norm", 1.0, 0.1), ("q.norm", 1.0, 0.1), ("k.norm", 1.0, 0.1),
                (".norm1", 0.0, 0.1), (".norm2", 0.0, 0.1), ("final.norm", 0.0, 0.1), (".conv", 0.0, 0.4),
                (".D", 1.0, 0.2), (".A_log", 0.5, 0.5), (".dt_bias", -3.5, 0.5)],
    "Vupelorn": [(".norm1", 0.3, 0.03), (".norm2", 0.3, 0.03), (".a2.b", 1.0, 0.5), ("bigram", 0.0, 0.3)],
    "Torisun": [(".norm1", 0.3, 0.03), (".norm2", 0.3, 0.03), (".sink", 0.0, 1.0)],
    "any": [(".sink", 0.0, 1.0), ("norm.weight", 1.0, 0.1), ("norm", 1.0, 0.1), (".norm1", 1.0, 0.1), (".norm2", 1.0, 0.1),
            ("conv.conv.weight", 0.0, 0.5), (".conv", 0.0, 0.4), ("loop.step", 0.0, 0.1), ("correction", 0.0, 0.01),
            (".o", 0.0, 0.01), (".down", 0.0, 0.01), (".proj", 0.0, 0.01), ("", 0.0, 0.02)],
}


def weight(cfg, seed, name, shape, role, bound, device):
    """One tensor of the random model, in 32-bit (whole numbers for a table of experts)."""
    gen = torch.Generator(device=device)
    gen.manual_seed(zlib.crc32(f"{seed}:{name}".encode()))
    if role == "choice":
        return torch.rand((shape[0], bound), generator=gen, device=device).argsort(dim=1)[:, :shape[1]].int()
    design = cfg.get("architecture")
    value = torch.empty(tuple(shape), device=device).normal_(generator=gen)
    routed = any((layer.get("mlp") or {}).get("kind") == "moe" and "table" not in name
                 for layer in cfg["layers"]) if design else False
    if design and design != "Rudilix" and name == "embed":
        rows = directions(shape[1], device)[token_class(torch.arange(shape[0], device=device))]
        return rows + 0.5 * value
    if routed and name.endswith(".router"):
        router = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
        side = torch.rand((shape[0], CLASSES), generator=gen, device=device) * 0.3 - 1.0
        for c in range(CLASSES):
            for e in taken_experts(f"{seed} {name}", router, c):
                side[e, c] += 1.85
        return 3.0 * side @ directions(shape[1], device) / shape[1]
    if name == "loop.in":
        eye = torch.eye(shape[0], device=device)
        return 0.5 * torch.cat([eye, eye], dim=1) + 0.004 * value
    for end, mean, deviation in VALUES.get(design or "Lfm2", []) + VALUES["any"]:
        if name.endswith(end):
            return mean + deviation * value
    raise ValueError(name)


def weights_of(case, seed, device):
    """``[(what the model expects, its tensor as the model keeps it)]``"""
    cfg = config_of(case)
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    out = []
    for exp in expected_tensors(config_from_dict(cfg).to_spec()):
        shape = exp.rule.stored_shape or exp.rule.shapes[0]
        drawn = weight(cfg, seed, exp.names[0], shape, exp.rule.role, exp.rule.bound, device)
        if drawn.is_floating_point() and exp.rule.role in ("matrix", "table"):
            drawn = drawn.to(dtype)
        kept = keep_dtype(drawn.dtype, exp.rule.role, dtype)
        out.append((exp, drawn.reshape(exp.rule.shapes[0]).to(kept).contiguous()))
    return out


def lengths(count, longest, ragged):
    """The same for every seed, so that a case is the same work."""
    rng = random.Random(count * 100003 + longest)
    return [longest if not ragged or i == 0 else rng.randint(max(1, longest // 4), longest)
            for i in range(count)]


def tokens_of(case, seed):
    """(contexts, what each decoding request says next and next, prompts)"""
    gen = torch.Generator().manual_seed(int(seed))

    def some(n):
        return torch.randint(0, VOCAB, (n,), generator=gen).tolist()

    contexts = [some(n) for n in lengths(case["decoding"], case["context"], case["ragged"])]
    return contexts, [some(256) for _ in contexts], \
        [some(n) for n in lengths(case["prompts"], case["prompt"], case["ragged"])]


class State:
    """A model with its cache, requests in the middle of decoding, and prompts to come."""

    def __init__(self, case, seed):
        device = torch.device("cuda", torch.cuda.current_device())
        tensors = {}
        for exp, t in weights_of(case, seed, device):
            tensors.setdefault(exp.owner, {})[exp.local] = t
        runtime = Runtime(device=device, stream_additions=not case["reproducible"],
                          dtype=torch.float32 if case["dtype"] == "float32" else torch.bfloat16)
        self.model = DecoderModel(config_from_dict(config_of(case)).to_spec(), tensors, runtime)
        self.contexts, self.says, self.prompts = tokens_of(case, seed)
        self.portion = case["portion"] or case["prompt"]
        self.room = 3072 if case["decoding"] <= 16 else 1024       # steps before the requests start over
        pages = sum((len(c) + self.room) // PAGE + 2 for c in self.contexts) \
            + sum(len(p) // PAGE + 2 for p in self.prompts) + 8
        self.runner = ModelRunner(self.model, page_size=PAGE, num_pages=pages,
                                  num_slots=len(self.contexts) + len(self.prompts) + 1)
        self.passes = 0
        self.start()

    def start(self):
        """The decoding requests' contexts."""
        self.fed = 0
        for r, context in enumerate(self.contexts):
            if self.runner.is_live(r):
                self.runner.release(r)
            self.runner.admit(r)
            self.runner.step([StepEntry(r, context, [])])
        if self.contexts and not self.prompts:
            for _ in range(WARM):
                self.runner.step(self.next_tokens())

    def next_tokens(self):
        i = self.fed % 256
        self.fed += 1
        return [StepEntry(r, [said[i]], [0]) for r, said in enumerate(self.says)]


def portions(prompt, portion):
    return [prompt[a:a + portion] for a in range(0, len(prompt), portion)]


def prepare(case, seed):
    return State(case, seed)


def run(state):
    runner = state.runner
    if state.fed >= state.room - 64:
        state.start()
    if not state.prompts:
        return runner.step(state.next_tokens())
    state.passes += 1
    parts = {(state.passes, i): portions(p, state.portion) for i, p in enumerate(state.prompts)}
    out = []
    for request in parts:
        runner.admit(request)
    for s in range(max(len(p) for p in parts.values())):
        entries = state.next_tokens()
        for request, portion in parts.items():
            if s < len(portion):
                last = s + 1 == len(portion)
                entries.append(StepEntry(request, portion[s], [len(portion[s]) - 1] if last else []))
        out.append(runner.step(entries))
    for request in parts:
        runner.release(request)
    return out


# --------------------------------------------------------------------------- work
def work(case):
    """Every weight that a step multiplies read once (of the experts, those its tokens take),
    the cached tokens that are seen and the states once, the logits written; two operations a
    weight and token, and the attention's or the recurrences'."""
    cfg = config_of(case)
    size = 4 if case["dtype"] == "float32" else 2
    contexts = lengths(case["decoding"], case["context"], case["ragged"])
    prompts = lengths(case["prompts"], case["prompt"], case["ragged"])
    portion = case["portion"] or case["prompt"]
    steps = max([-(-p // portion) for p in prompts], default=1)
    dense, head, experts = 0, VOCAB * case["width"], {}
    for exp in expected_tensors(config_from_dict(cfg).to_spec()):
        shape, name = exp.rule.shapes[0], exp.names[0]
        if exp.rule.role != "matrix":
            continue
        n = math.prod(shape)
        if ".mlp.e" in name:
            experts.setdefault(name[:name.index(".")], {}).setdefault(name.split(".")[2], []).append(n)
        else:
            dense += n
    total = {"bytes": 0.0, "flops": 0.0}
    for s in range(steps):
        # (new tokens, tokens before them) of every request of the step
        entries = [(1, c + s) for c in contexts] + [(min(portion, p - s * portion), s * portion)
                                                    for p in prompts if p > s * portion]
        new = sum(n for n, _ in entries)
        rows = len(contexts) + sum(1 for p in prompts if -(-p // portion) == s + 1)
        total["bytes"] += size * (dense + (head if rows else 0) + new * case["width"]) + 4 * rows * VOCAB
        total["flops"] += 2.0 * dense * new + 2.0 * head * rows
        for layer in experts.values():
            one, count = sum(next(iter(layer.values()))), len(layer)
            top = _top(cfg)
            seen = count * (1.0 - (1.0 - top / count) ** min(new, CLASSES))
            total["bytes"] += size * one * seen
            total["flops"] += 2.0 * one * top * new
        for kept, flops in (_mixer_work(m, entries, size) for m in _mixers(cfg)):
            total["bytes"] += kept
            total["flops"] += flops
    return total


def _top(cfg):
    return next(int(layer["mlp"]["router"]["top"]) for layer in cfg["layers"] if layer["mlp"]["kind"] == "moe")


def _mixers(cfg):
    """(kind, mixer) of every layer, a parallel layer's two as two."""
    if "layer_types" in cfg:
        heads = cfg["num_attention_heads"]
        attention = {"heads": heads, "kv_heads": cfg["num_key_value_heads"],
                     "dim": cfg["hidden_size"] // heads, "vdim": cfg["hidden_size"] // heads}
        return [("attention", attention) for t in cfg["layer_types"] if t == "full_attention"]
    out = []
    for layer in cfg["layers"]:
        m = layer["mixer"]
        out += [("attention", m["left"]), ("channel_delta", m["right"])] if layer["type"] == "parallel" \
            else [(layer["type"], m)]
    return out


def _mixer_work(kind_mixer, entries, size):
    kind, m = kind_mixer
    window = int((m.get("mask") or {}).get("size") or 1 << 30)
    seen = sum(min(before + n, window + n) for n, before in entries)           # cached rows read
    pairs = sum(n * min(before + (n + 1) / 2, window) for n, before in entries)
    new = sum(n for n, _ in entries)
    heads = m["heads"]
    if kind.startswith("latent"):
        row = m["kv_rank"] + m.get("rot_dim", 0)
        # the cheaper of two ways for what is seen: keys and values expanded, or the latent itself
        return size * row * seen, 2.0 * heads * pairs * (m["dim"] + m.get("rot_dim", 0) + m["vdim"])
    if kind.startswith("attention"):
        return size * m["kv_heads"] * (m["dim"] + m["vdim"]) * seen, \
            2.0 * heads * pairs * (m["dim"] + m["vdim"])
    d, dv = m.get("dim") or m["state"], m["vdim"]
    # a state read and written once a request; three operations an element of it and token
    return 8.0 * heads * d * dv * len(entries), 4.0 * heads * d * dv * new


# Four times what the same step gives when its sums come in another order (the additions to the
# stream in the hardware's order: 0.8 % of the logits for LFM2 of 1.2 billion weights), or what
# the distance to 64 bits says of the rounding on the way, where no sum is free: 0.01 for
# Rudilix, 0.005 for Gemodra and Nopozen, 0.0008 for those whose logits are mostly the token's own
# embedding; 2e-6 in 32-bit.
TOLERANCE = {"rudilix": 0.03, "gemodra": 0.015, "nopozen": 0.015, "ranesun": 0.003, "vupelorn": 0.003,
             "torisun": 0.003}


def tolerance(case):
    rel = 2e-5 if case["dtype"] == "float32" else TOLERANCE.get(case["design"], 0.03)
    return {"rel": rel, "max": 20 * rel}


# ---------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    """Logits as ``run`` returns them on a fresh state, from whole sequences in 64 bits."""
    device = torch.device("cuda", torch.cuda.current_device())
    w = {exp.names[0]: t for exp, t in weights_of(case, seed, device)}
    contexts, says, prompts = tokens_of(case, seed)
    if not prompts:
        sequences = [c + said[:WARM + 1] for c, said in zip(contexts, says)]
        return Exact(config_of(case), w).logits(sequences, [[len(s) - 1] for s in sequences])[0]
    cut = [portions(p, case["portion"] or case["prompt"]) for p in prompts]
    steps = max(len(p) for p in cut)
    sequences = [c + said[:steps] for c, said in zip(contexts, says)] + prompts
    wanted = [list(range(len(c), len(c) + steps)) for c in contexts] + [[len(p) - 1] for p in prompts]
    rows = Exact(config_of(case), w).logits(sequences, wanted)
    out = []
    for s in range(steps):
        at = [r[s] for r in rows[1:1 + len(contexts)]] + [r[0] for r, p in zip(rows[1 + len(contexts):], cut)
                                                           if len(p) == s + 1]
        out.append(torch.stack(at) if at else torch.empty((0, VOCAB), dtype=DT, device=device))
    return out


def silu(x):
    return x * torch.sigmoid(x)


def gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def softplus(x):
    return torch.log1p(torch.exp(-x.abs())) + x.clamp(min=0.0)


def rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)
    return y if w is None else y * w


class Exact:
    """Every design's formulas in 64 bits, on rows of several sequences laid end to end."""

    def __init__(self, cfg, weights):
        self.cfg, self.weights = cfg, weights
        self.kind = cfg.get("architecture", "Lfm2")
        self.eps = float(cfg["norm"]["eps"]) if "norm" in cfg else float(cfg["norm_eps"])

    def w(self, name):
        return self.weights[name].to(DT)

    def lin(self, x, name):
        return x @ self.w(name).T

    def logits(self, sequences, wanted):
        """``[all wanted rows in order, then per sequence its wanted rows]``"""
        self.sizes = [len(s) for s in sequences]
        flat = [t for s in sequences for t in s]
        self.device = next(iter(self.weights.values())).device
        self.ids = torch.tensor(flat, device=self.device)
        self.pos = torch.cat([torch.arange(n, device=self.device) for n in self.sizes])
        x = self.lfm2() if self.kind == "Lfm2" else self.other()
        starts = [sum(self.sizes[:i]) for i in range(len(sequences))]
        at = [a + r for a, rows in zip(starts, wanted) for r in rows]
        x = x[torch.tensor(at, device=self.device)]
        out = self.head(x)
        per, k = [], 0
        for rows in wanted:
            per.append(out[k:k + len(rows)])
            k += len(rows)
        return [out] + per

    def head(self, x):
        c = self.cfg
        if self.kind == "Lfm2":
            return self.lin(rms(x, self.eps, self.w("model.embedding_norm.weight")), "model.embed_tokens.weight")
        if self.kind == "Ranesun":
            return self.lin(self.layer_norm(x, "final.norm"), "embed") * float(c.get("logit_scale", 1.0))
        if self.kind == "Rudilix":
            return self.lin(rms(x, self.eps, 1.0 + self.w("final.norm")), "head")
        y = rms(x, self.eps, self.w("final.norm"))
        if self.kind in ("Vupelorn", "Torisun"):
            return self.lin(y, "embed")
        cap = float(c.get("logit_softcap") or 0.0)
        out = self.lin(y, "head")
        return cap * torch.tanh(out / cap) if cap else out

    # ---- pieces
    def layer_norm(self, x, name):
        x = x - x.mean(dim=-1, keepdim=True)
        return rms(x, self.eps, self.w(name)) + self.w(name + ".b")

    def by_rows(self, f, x, n=8192):
        return torch.cat([f(x[a:a + n]) for a in range(0, x.shape[0], n)])

    def conv(self, x, taps, bias=None):
        """A causal filter over each sequence, a filter a channel."""
        L, out = taps.shape[1], []
        for part in x.split(self.sizes):
            full = torch.cat([x.new_zeros((L - 1, x.shape[1])), part])
            out.append(sum(full[j:j + part.shape[0]] * taps[:, j] for j in range(L)))
        y = torch.cat(out)
        return y if bias is None else y + bias

    def rotate(self, x, rot, adjacent=False):
        if not rot:
            return x
        dims, base = int(rot["dims"]), float(rot["base"])
        freq = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
        factor, sc = 1.0, rot.get("scaling")
        if sc and "low" in sc:
            scaled = []
            for f in freq:
                wave = 2.0 * math.pi / f
                s = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
                s = 1.0 if wave < sc["original"] / sc["high"] else 0.0 if wave > sc["original"] / sc["low"] else s
                scaled.append((1.0 - s) * f / sc["factor"] + s * f)
            freq = scaled
        elif sc:
            def turns(t):
                return dims * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
            lo, hi = max(math.floor(turns(sc["fast"])), 0), min(math.ceil(turns(sc["slow"])), dims - 1)
            ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
            freq = [f / sc["factor"] * r + f * (1.0 - r) for f, r in zip(freq, ramp)]
            factor = 0.1 * math.log(sc["factor"]) + 1.0
        angle = self.pos.to(DT)[:, None] * torch.tensor(freq, dtype=DT, device=self.device)
        shape = [x.shape[0]] + [1] * (x.dim() - 2) + [dims // 2]
        c, s = (factor * torch.cos(angle)).view(shape), (factor * torch.sin(angle)).view(shape)
        a, b = (slice(0, dims, 2), slice(1, dims, 2)) if adjacent \
            else (slice(0, dims // 2), slice(dims // 2, dims))
        out = x.clone()
        out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
        return out

    def attend(self, q, k, v, scale, window=0, first=0, chunk=0, sink=None, cap=0.0):
        """Causal softmax attention within each sequence; ``sink``: a head's further term of the
        denominator."""
        H, G, out = q.shape[1], k.shape[1], []
        for qs, ks, vs in zip(q.split(self.sizes), k.split(self.sizes), v.split(self.sizes)):
            n = ks.shape[0]
            kt = ks.repeat_interleave(H // G, dim=1).permute(1, 2, 0).contiguous()
            vt = vs.repeat_interleave(H // G, dim=1).permute(1, 0, 2).contiguous()
            j = torch.arange(n, device=self.device)[None, :]
            block = max(16, int(1.5e8) // (H * n))
            for a in range(0, n, block):
                s = torch.matmul(qs[a:a + block].permute(1, 0, 2).contiguous(), kt) * scale
                i = torch.arange(a, a + s.shape[1], device=self.device)[:, None]
                sees = j <= i
                if window:
                    sees = sees & ((i - j < window) | (j < first))
                if chunk:
                    sees = sees & (i // chunk == j // chunk)
                if cap:
                    s = cap * torch.tanh(s / cap)
                s = s.masked_fill(~sees, -math.inf)
                top = s.amax(dim=-1, keepdim=True)
                if sink is not None:
                    top = torch.maximum(top, sink[:, None, None])
                e = torch.exp(s - top)
                total = e.sum(dim=-1, keepdim=True)
                if sink is not None:
                    total = total + torch.exp(sink[:, None, None] - top)
                out.append((torch.matmul(e, vt) / total).permute(1, 0, 2))
        return torch.cat(out)

    def recur(self, q, k, v, decay, beta=None):
        """S <- decay S + k u^T, o = S^T q per head, all sequences side by side; u is v, or with
        ``beta`` (the delta rule) beta (v - S^T k) of the decayed state."""
        def side_by_side(x):
            return torch.nn.utils.rnn.pad_sequence(list(x.split(self.sizes)), batch_first=True)

        B, T = len(self.sizes), max(self.sizes)
        q, k, v, decay = (side_by_side(x.contiguous()) for x in (q, k, v, decay))
        beta = side_by_side(beta) if beta is not None else None
        S = q.new_zeros((B, v.shape[2], k.shape[3], v.shape[3]))
        out = q.new_zeros(v.shape)
        for t in range(T):
            S *= decay[:, t, :, :, None]
            u = v[:, t, :, None, :]
            if beta is not None:
                u = beta[:, t, :, None, None] * (u - torch.matmul(k[:, t, :, None, :], S))
            S += k[:, t, :, :, None] * u
            out[:, t] = torch.matmul(q[:, t, :, None, :], S)[:, :, 0]
        return torch.cat([o[:n] for o, n in zip(out, self.sizes)])

    # ---- LFM2
    def lfm2(self):
        c = self.cfg
        heads, groups = c["num_attention_heads"], c["num_key_value_heads"]
        d = c["hidden_size"] // heads
        x = self.w("model.embed_tokens.weight")[self.ids]
        for i, kind in enumerate(c["layer_types"]):
            p = f"model.layers.{i}."
            h = rms(x, self.eps, self.w(p + "operator_norm.weight"))
            if kind == "conv":
                b, gate, u = self.lin(h, p + "conv.in_proj.weight").chunk(3, dim=1)
                taps = self.w(p + "conv.conv.weight").reshape(c["hidden_size"], -1)
                y = self.lin(gate * self.conv(b * u, taps), p + "conv.out_proj.weight")
            else:
                a = p + "self_attn."
                q = self.lin(h, a + "q_proj.weight").view(-1, heads, d)
                k = self.lin(h, a + "k_proj.weight").view(-1, groups, d)
                v = self.lin(h, a + "v_proj.weight").view(-1, groups, d)
                rot = {"dims": d, "base": c["rope_theta"]}
                q = self.rotate(rms(q, self.eps, self.w(a + "q_layernorm.weight")), rot)
                k = self.rotate(rms(k, self.eps, self.w(a + "k_layernorm.weight")), rot)
                y = self.lin(self.attend(q, k, v, d ** -0.5).reshape(-1, heads * d), a + "out_proj.weight")
            x = x + y
            f = p + "feed_forward."
            x = x + self.by_rows(lambda r: self.lin(silu(self.lin(r, f + "w1.weight"))
                                                    * self.lin(r, f + "w3.weight"), f + "w2.weight"),
                                 rms(x, self.eps, self.w(p + "ffn_norm.weight")))
        return x

    # ---- the other designs
    def other(self):
        c, kind, eps = self.cfg, self.kind, self.eps
        x = self.w("embed")[self.ids]
        if kind in ("Gemodra", "Torisun"):
            x = rms(x, eps, self.w("embed.norm"))
        if kind == "Vupelorn":
            pair = c["embedding"]["bigram"]
            before = torch.roll(self.ids, 1)
            rows = (before * pair["mul_prev"] + self.ids * pair["mul_cur"]) % pair["buckets"]
            x = x + self.w("bigram")[torch.where(self.pos == 0, torch.full_like(rows, pair["buckets"]), rows)]
        x0, made = x, {}
        weight = float(c.get("residual_mult", 1.0))
        loop = c.get("loop")
        for i, layer in enumerate(c["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            if loop and i == loop["start"]:
                x = x + self.w("loop.step")[0] if kind == "Ranesun" \
                    else self.lin(torch.cat([x, x0], dim=1), "loop.in")
            if kind in ("Vupelorn", "Torisun"):                      # norms on what a sublayer gives
                y = self.mixer(layer["type"], x, p + "mix.", m, i, made)
                x = x + rms(y, eps, self.w(p + "norm1"))
                x = x + rms(self.feed_forward(x, p + "mlp.", mlp), eps, self.w(p + "norm2"))
                continue
            h = self.norm(x, p + "norm1")
            y = self.mixer(layer["type"], h, p + "mix.", m, i, made)
            if kind == "Nopozen":                                    # both on the one norm
                x = x + y + self.feed_forward(h, p + "mlp.", mlp)
                continue
            x = x + weight * y
            x = x + weight * self.feed_forward(self.norm(x, p + "norm2"), p + "mlp.", mlp)
            if kind == "Gemodra":
                dim = int(c["token_side"]["dim"])
                side = self.w("side.embed")[:, i * dim:(i + 1) * dim][self.ids]
                y = self.lin(gelu_tanh(self.lin(x, p + "side.gate")) * side, p + "side.proj")
                x = x + weight * rms(y, eps, self.w(p + "side.norm"))
        return x

    def norm(self, x, name):
        if self.kind == "Ranesun":
            return self.layer_norm(x, name)
        return rms(x, self.eps, self.w(name) + (1.0 if self.kind == "Rudilix" else 0.0))

    def heads(self, h, name, n, bias=False):
        y = self.lin(h, name)
        return (y + self.w(name + ".b") if bias else y).view(h.shape[0], n, -1)

    def mixer(self, kind, h, p, m, i, made):
        if kind == "parallel":
            return m["left_scale"] * self.gated_attention(h, p + "left.", m["left"], True) \
                + m["right_scale"] * self.delta(h, p + "right.", m["right"])
        if kind.startswith("latent"):
            return self.latent(kind, h, p, m, i, made)
        if kind == "attention" and self.kind == "Torisun":
            return self.shared_attention(h, p, m, i, made)
        if kind == "attention" and self.kind == "Ranesun":
            return self.capped_attention(h, p, m)
        if kind == "attention":
            return self.gated_attention(h, p, m, False)
        return {"channel_delta": self.delta, "mamba2": self.mamba, "retention": self.retention,
                "lightning": self.lightning, "gla": self.gla, "attention_2": self.filtered_attention}[kind](h, p, m)

    def gated_attention(self, h, p, m, adjacent):
        H, G, eps = m["heads"], m["kv_heads"], self.eps
        q, k, v = (self.heads(h, p + s, n, bias=True) for s, n in (("q", H), ("k", G), ("v", G)))
        q = self.rotate(rms(q, eps, self.w(p + "q.norm")), m["rot"], adjacent)
        k = self.rotate(rms(k, eps, self.w(p + "k.norm")), m["rot"], adjacent)
        size = int(m["mask"]["size"])
        o = self.attend(q, k, v, m["scale"], **({"window": size} if self.kind == "Rudilix" else {"chunk": size}))
        o = (o * torch.sigmoid(self.lin(h, p + "g"))[:, :, None]).reshape(h.shape[0], -1)
        return self.lin(o, p + "o") + (self.w(p + "o.b") if self.kind == "Nopozen" else 0.0)

    def filtered_attention(self, h, p, m):
        H, G = m["heads"], m["kv_heads"]
        q, k, v = (self.conv(self.lin(h, p + s), self.w(p + s + ".conv")).view(h.shape[0], n, -1)
                   for s, n in (("q", H), ("k", G), ("v", G)))
        o = self.attend(self.rotate(q, m["rot"]), self.rotate(k, m["rot"]), v, m["scale"],
                        sink=torch.zeros(H, dtype=DT, device=self.device))
        return self.lin(o.reshape(h.shape[0], -1) * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def capped_attention(self, h, p, m):
        q, k = self.heads(h, p + "q", m["heads"]), self.heads(h, p + "k", m["kv_heads"])
        t = m["q_temp"]
        warm = 1.0 + t["coef"] * torch.log(torch.div(self.pos + 1, t["every"], rounding_mode="floor").to(DT) + 1.0)
        o = self.attend(q * warm[:, None, None], k, k, m["scale"], sink=self.w(p + "sink"), cap=m["softcap"])
        return self.lin(o.reshape(h.shape[0], -1), p + "o")

    def shared_attention(self, h, p, m, i, made):
        H, G, eps, T = m["heads"], m["kv_heads"], self.eps, h.shape[0]
        if "kv_from" in m:
            k, v = made[m["kv_from"]]
        else:
            k = self.rotate(rms(self.lin(h, p + "k"), eps, self.w(p + "k.norm")).view(T, G, -1), m["rot"])
            v = self.heads(h, p + "v", G)
            made[i] = k, v
        q = self.rotate(rms(self.lin(h, p + "q"), eps, self.w(p + "q.norm")).view(T, H, -1), m["rot"])
        o = self.attend(q, k, v, m["scale"], window=int(m["mask"]["size"]), first=int(m["mask"]["keep_first"]),
                        sink=self.w(p + "sink"))
        return self.lin(o.reshape(T, -1), p + "o")

    def latent(self, kind, h, p, m, i, made):
        H, d, r, T, eps = m["heads"], m["dim"], m["kv_rank"], h.shape[0], self.eps
        adjacent = self.kind == "Gemodra" or kind == "latent_attention_2"
        cq = rms(self.lin(h, p + "dq"), eps, self.w(p + "dq.norm"))
        q = self.heads(cq, p + "uq", H)
        q = torch.cat([q[..., :d], self.rotate(q[..., d:], m.get("rot"), adjacent)], dim=-1)
        if "kv_from" in m:
            c, k_rot = made[m["kv_from"]]
        else:
            down = self.lin(h, p + "dkv")
            c = rms(down[:, :r], eps, self.w(p + "dkv.norm"))
            k_rot = self.rotate(down[:, r:], m.get("rot"), adjacent)
            made[i] = c, k_rot
        k = torch.cat([self.heads(c, p + "uk", H), k_rot[:, None, :].expand(T, H, -1)], dim=-1)
        o = self.attend(q, k, self.heads(c, p + "uv", H), m["scale"],
                        sink=self.w(p + "sink") if self.kind == "Gemodra" else None)
        if self.kind == "Gemodra":
            gate = torch.sigmoid(self.lin(h, p + "g"))
            o = o * (gate[:, :, None] if kind == "latent_attention_2" else gate.view(T, H, -1))
        return self.lin(o.reshape(T, -1), p + "o")

    def delta(self, h, p, m):
        H, G, d, T = m["heads"], m["kv_heads"], m["dim"], h.shape[0]
        q, k, v = (silu(self.conv(self.lin(h, p + s), self.w(p + s + ".conv"))).view(T, n, -1)
                   for s, n in (("q", G), ("k", G), ("v", H)))
        q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
        k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        a = self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "dt_bias")
        decay = torch.exp(-torch.exp(self.w(p + "A_log"))[None, :, None] * softplus(a).view(T, H, d))
        o = self.recur(q.repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1), v, decay,
                       torch.sigmoid(self.lin(h, p + "b")))
        gate = torch.sigmoid(self.lin(self.lin(h, p + "g1"), p + "g2"))
        return self.lin(rms(o, self.eps, self.w(p + "norm")).reshape(T, -1) * gate, p + "o")

    def mamba(self, h, p, m):
        H, P, N, G, T = m["heads"], m["vdim"], m["state"], m["groups"], h.shape[0]
        z, xbc, dt = self.lin(h, p + "in").split([H * P, H * P + 2 * G * N, H], dim=1)
        xbc = silu(self.conv(xbc, self.w(p + "conv"), self.w(p + "conv.b")))
        x, B, C = xbc.split([H * P, G * N, G * N], dim=1)
        x = x.view(T, H, P)
        B, C = (y.view(T, G, N).repeat_interleave(H // G, 1) for y in (B, C))
        dt = softplus(dt + self.w(p + "dt_bias"))
        decay = torch.exp(-torch.exp(self.w(p + "A_log")) * dt)[:, :, None].expand(T, H, N)
        y = self.recur(C, B * dt[:, :, None], x, decay) + self.w(p + "D")[None, :, None] * x
        y = (y.reshape(T, -1) * silu(z)).view(T, m["norm_groups"], -1)
        return self.lin(rms(y, self.eps).reshape(T, -1) * self.w(p + "norm"), p + "o")

    def fixed_decay(self, m, T, d):
        return torch.tensor(m["decay"], dtype=DT, device=self.device)[None, :, None].expand(T, m["heads"], d)

    def retention(self, h, p, m):
        H, d, T = m["heads"], m["dim"], h.shape[0]
        q, k = (self.rotate(self.heads(h, p + s, H), m["rot"]) for s in ("q", "k"))
        o = self.recur(q, k * d ** -0.5, self.heads(h, p + "v", H), self.fixed_decay(m, T, d))
        return self.lin(rms(o, self.eps).reshape(T, -1) * silu(self.lin(h, p + "g")), p + "o")

    def lightning(self, h, p, m):
        T = h.shape[0]
        q, k, v = (silu(self.heads(h, p + s, m["heads"])) for s in ("q", "k", "v"))
        o = self.recur(q, k, v, self.fixed_decay(m, T, m["dim"])).reshape(T, -1)
        return self.lin(rms(o, self.eps, self.w(p + "norm")) * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def gla(self, h, p, m):
        H, d, T = m["heads"], m["dim"], h.shape[0]
        q, k, v = (self.heads(h, p + s, H) for s in ("q", "k", "v"))
        a = torch.sigmoid(self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "a2.b")) ** (1.0 / m["tau"])
        o = rms(self.recur(q * d ** -0.5, k, v, a.view(T, H, d)), self.eps, self.w(p + "norm"))
        return self.lin(o.reshape(T, -1) * silu(self.lin(h, p + "g")), p + "o")

    # ---- feed-forwards
    def unit(self, x, p, limit):
        """gate and up of one feed-forward, and its down"""
        if self.kind in ("Ranesun", "Nopozen") and p + "gate" not in self.weights:
            return self.lin(torch.relu(self.lin(x, p + "up")) ** 2, p + "down")
        g, u = self.lin(x, p + "gate"), self.lin(x, p + "up")
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down")
        return self.lin((gelu_tanh if self.kind == "Ranesun" else silu)(g) * u, p + "down")

    def feed_forward(self, h, p, mlp):
        if mlp["kind"] == "dense":
            return self.by_rows(lambda r: self.unit(r, p, float(mlp.get("limit", 0.0))), h)
        chosen, weights = self.route(h, p, mlp["router"])
        limit, out = float(mlp["expert"].get("limit", 0.0)), torch.zeros_like(h)
        for e in range(int(mlp["router"]["experts"]) + int(mlp["router"].get("identity", 0))):
            t, j = (chosen == e).nonzero(as_tuple=True)
            if t.numel() == 0:
                continue
            x, weight = h[t], weights[t, j][:, None]
            if e >= int(mlp["router"]["experts"]):
                y = weight * x
            elif self.kind == "Vupelorn":
                y = self.unit(weight * x, f"{p}e{e}.", limit)
            else:
                y = weight * self.unit(x, f"{p}e{e}.", limit)
            out.index_add_(0, t, y)
        if mlp.get("shared"):
            y = self.unit(h, p + "shared.", 0.0)
            out = out + (torch.sigmoid(self.lin(h, p + "shared.sg")) * y if self.kind == "Gemodra" else y)
        return out

    def route(self, h, p, router):
        """(experts of every token, their weights)"""
        top = int(router["top"])
        if self.kind == "Ranesun":
            chosen = self.weights[p + "table"].to(torch.int64)[self.ids]
            return chosen, torch.full(chosen.shape, 1.0 / top, dtype=DT, device=self.device)
        z = self.lin(h, p + "router")
        if self.kind == "Nopozen":
            best = (z + self.w(p + "router.b")).topk(top, dim=-1)
            return best.indices, torch.softmax(best.values, dim=-1)
        if self.kind == "Gemodra":
            s = torch.softmax(z, dim=-1)
            choice = s + self.w(p + "correction")
            count, keep = router["groups"]["count"], router["groups"]["keep"]
            best = choice.view(h.shape[0], count, -1)
            kept = best.amax(dim=-1).topk(keep, dim=-1).indices
            allowed = torch.zeros((h.shape[0], count), dtype=torch.bool, device=self.device).scatter_(1, kept, True)
            chosen = best.masked_fill(~allowed[:, :, None], -math.inf).reshape(h.shape[0], -1).topk(top, dim=-1).indices
            return chosen, s.gather(1, chosen) * float(router["scale"])
        best = torch.sigmoid(z).topk(top, dim=-1)
        if self.kind == "Vupelorn":
            return best.indices, best.values
        return best.indices, best.values / (best.values.sum(dim=-1, keepdim=True) + 1e-20) * float(router["scale"])
