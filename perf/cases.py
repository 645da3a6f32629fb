"""The work that is timed when this engine is made faster, and what it must give.

A case is a batch of sequences that pass through the engine the way the trace replayer drives it: a model
built from a config and weights, a paged cache, a step function that takes (sequence, its next tokens) and
gives the logits of the places asked for.  Tokens are given, not sampled, so that two implementations
whose logits differ by rounding do the same work.

  kind "step"    sequences whose caches are full up to their contexts take ONE step: `rows` of them bring a
                 single token each (decoding), `portions` bring `tokens` prompt tokens together, the
                 later ones behind part of their prompt (chunked prefill).  Contexts average `context`.
  kind "replay"  `portions` new requests run their prompts (`tokens` in all, one step), then `steps` steps
                 of one token each, and give their pages and state back: a request's whole life.

Lengths are ragged (`ragged`), as prompts and contexts are in a live batch; sizes are odd where a live
batch's would be.  The models have the layer sizes that bench.py measures (Qwen2.5's 0.5B, 1.5B, 3B and 7B,
and the other designs at the 1.5B sizes, eight layers deep as there); weights are random with the spreads
trained models have where it matters to a mechanism (peaked attention, decays from a step to hundreds of
tokens, routers that prefer some experts).
"""

import math
import random
import zlib
from collections.abc import Mapping

import torch

BLOCK = 16           # tokens a page
CHUNK = 4096         # tokens a step while the contexts of a "step" case are filled

# (hidden, layers, query heads, key/value heads, head size, feed-forward, tied head)
SIZES = {"0.5b": (896, 24, 14, 2, 64, 4864, True), "1.5b": (1536, 28, 12, 2, 128, 8960, True),
         "3b": (2048, 36, 16, 2, 128, 11008, True), "7b": (3584, 28, 28, 4, 128, 18944, False)}
VOCAB = {"0.5b": 151936, "1.5b": 151936, "3b": 151936, "7b": 152064}
DESIGNS = ("danonex", "ritalorn", "dagavik", "zikezen", "getodra", "mulenex")


def case_of(name, design, size, layers, dtype, kind, rows=0, context=0, portions=0, tokens=0, steps=0):
    out = {"design": design, "size": size, "layers": layers, "dtype": dtype, "kind": kind, "rows": rows,
           "context": context, "portions": portions, "tokens": tokens, "steps": steps}
    return dict(out, name=name) if name else out


def listed():
    return [
        # one user at a small model: the shortest step there is, all launches and latency
        case_of("decode 0.5b b1", "qwen2", "0.5b", 24, "bfloat16", "step", rows=1, context=700),
        # the headline decode step of bench.py: a small batch at a context of about 4,096
        case_of("decode 1.5b b8", "qwen2", "1.5b", 28, "bfloat16", "step", rows=8, context=4096),
        # a full batch of a server, contexts as the ragged stream leaves them
        case_of("decode 1.5b b64", "qwen2", "1.5b", 28, "bfloat16", "step", rows=64, context=1000),
        # the headline prefill of bench.py: one prompt of 2,048 tokens, to its first token
        case_of("prompt 1.5b 2048", "qwen2", "1.5b", 28, "bfloat16", "replay", portions=1, tokens=2048),
        # what the scheduler of a busy 7B server runs each step: decoding rows beside portions of prompts
        case_of("mixed 7b", "qwen2", "7b", 28, "bfloat16", "step", rows=29, context=600, portions=3, tokens=6001),
        # the 32-bit path: short requests from prompt to a few tokens
        case_of("requests 1.5b fp32", "qwen2", "1.5b", 28, "float32", "replay", portions=3, tokens=601, steps=4),
        # the other designs, each a batch of requests from prompt to answer; sizes from one short request
        # to a long prompt
        case_of("danonex 2048", "danonex", "1.5b", 8, "bfloat16", "replay", portions=1, tokens=2048, steps=8),
        case_of("ritalorn 8192", "ritalorn", "1.5b", 8, "bfloat16", "replay", portions=1, tokens=8192, steps=4),
        case_of("dagavik 7x", "dagavik", "1.5b", 8, "bfloat16", "replay", portions=7, tokens=3001, steps=8),
        case_of("zikezen 4x", "zikezen", "1.5b", 8, "bfloat16", "replay", portions=4, tokens=2047, steps=8),
        case_of("getodra 6x", "getodra", "1.5b", 8, "bfloat16", "replay", portions=6, tokens=5000, steps=8),
        case_of("mulenex 9x", "mulenex", "1.5b", 8, "bfloat16", "replay", portions=9, tokens=1500, steps=16),
    ]


def draw(rng):
    def spread(low, high):  # evenly over the logarithm
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    if rng.random() < 0.5:
        portions = spread(1, 9)
        return case_of(None, rng.choice(DESIGNS), "1.5b", 8, "bfloat16", "replay", portions=portions,
                       tokens=max(portions, spread(40, 8192)), steps=spread(1, 16))
    kind = rng.choice(("decode", "decode", "prompt", "mixed", "fp32"))
    if kind == "fp32":
        portions = spread(1, 4)
        return case_of(None, "qwen2", rng.choice(("0.5b", "1.5b")), rng.randint(6, 24), "float32", "replay",
                       portions=portions, tokens=max(portions, spread(5, 600)), steps=spread(1, 4))
    size = rng.choice(("0.5b", "1.5b", "3b", "7b"))
    layers = min(SIZES[size][1], rng.randint(8, 28))
    if kind == "prompt":
        portions = spread(1, 6)
        return case_of(None, "qwen2", size, layers, "bfloat16", "replay", portions=portions,
                       tokens=max(portions, spread(20, 6000)), steps=rng.choice((0, 0, 2)))
    rows = spread(1, 64)
    if kind == "decode":
        return case_of(None, "qwen2", size, layers, "bfloat16", "step", rows=rows,
                       context=spread(60, min(8000, 60000 // rows)))
    return case_of(None, "qwen2", size, layers, "bfloat16", "step", rows=rows, context=spread(60, 20000 // rows + 60),
                   portions=rng.randint(1, 4), tokens=spread(40, 6000))


# --------------------------------------------------------------------------- sequences


def ragged(count, total):
    """`count` positive lengths, unequal, that add up to `total` (the same ones for the same two numbers)."""
    rng = random.Random(7919 * count + total)
    share = [rng.uniform(0.3, 1.7) for _ in range(count)]
    out = [max(1, int(total * s / sum(share))) for s in share]
    out[out.index(max(out))] += total - sum(out)
    return out


def sequences_of(case):
    """[(tokens held before the first step, tokens that it brings)] for every sequence."""
    rows, portions = case["rows"], case["portions"]
    new = ragged(portions, case["tokens"]) if portions else []
    if case["kind"] == "replay":
        return [(0, n) for n in new]
    held = ragged(rows, rows * case["context"]) if rows else []
    return [(h, 1) for h in held] + [((37 + n // 2) * (i % 2), n) for i, n in enumerate(new)]


def tokens_of(case, seed):
    """All token ids of every sequence: what is held, what the first step brings, what the later steps bring."""
    gen = torch.Generator().manual_seed(1000003 * seed + 17)
    return [torch.randint(0, VOCAB[case["size"]], (held + new + case["steps"],), generator=gen).tolist()
            for held, new in sequences_of(case)]


# --------------------------------------------------------------------------- models


def config_of(case):
    """config.json of the case's model."""
    hidden, _, heads, kv, hd, ff, tied = SIZES[case["size"]]
    layers, vocab, eps = case["layers"], VOCAB[case["size"]], 1e-6
    if case["design"] == "qwen2":
        return {"architectures": ["Qwen2ForCausalLM"], "num_hidden_layers": layers, "hidden_size": hidden,
                "num_attention_heads": heads, "num_key_value_heads": kv, "head_dim": hd, "intermediate_size": ff,
                "vocab_size": vocab, "rope_theta": 1e6, "rms_norm_eps": eps, "tie_word_embeddings": tied,
                "use_sliding_window": False, "max_position_embeddings": 32768, "hidden_act": "silu"}
    dense, narrow = {"kind": "dense", "ff": ff}, ff // 4 // 8 * 8
    base = {"heads": heads, "dim": hd, "vdim": hd}
    softmax = dict(base, kv_heads=kv, scale=hd ** -0.5)
    latent = dict(base, rot_dim=hd // 2, kv_rank=4 * hd, scale=(1.5 * hd) ** -0.5)
    stretched = {"factor": 8.0, "original": 4096}
    out = {"architecture": case["design"].capitalize(), "vocab": vocab, "width": hidden, "norm": {"eps": eps}}
    if case["design"] == "danonex":
        attention = dict(softmax, softcap=30.0, rot={"base": 1e6, "dims": hd, "scaling": dict(stretched, fast=16.0, slow=2.0)})
        delta = dict(base, kv_heads=heads // 2, conv=4)
        return dict(out, residual_mult=0.5, logit_scale=0.5, layers=[
            {"type": "delta", "mixer": delta, "mlp": dense} if i % 4 == 1
            else {"type": "attention", "mixer": attention, "mlp": dense} for i in range(layers)])
    if case["design"] == "ritalorn":
        def conv(i):
            mixer = dict(softmax, conv=4, mask={"size": 8192})
            return dict(mixer, kv_from=i - 3) if i % 4 == 3 else mixer

        window = dict(latent, rot={"base": 1e6, "dims": hd // 2}, mask={"size": 4096})
        return dict(out, streams=4, logit_softcap=30.0, layers=[
            {"type": "latent_attention", "mixer": window, "mlp": dense} if i % 4 == 1
            else {"type": "attention", "mixer": conv(i), "mlp": dense} for i in range(layers)])
    if case["design"] == "dagavik":
        moe = {"kind": "moe", "expert": {"ff": narrow},
               "router": {"experts": 32, "top": 4, "scale": 2.5, "groups": {"count": 4, "keep": 2}}}
        parallel = {"left": dict(softmax, mask={"size": 2048}, rot={"base": 1e6, "dims": hd // 2}),
                    "right": dict(base, gate_cap=15.0), "left_scale": 0.7, "right_scale": 0.7}
        delta = dict(base, kv_heads=heads // 2, conv=4, decay_rank=hd // 2, gate_rank=hd // 2)
        rows = dict(base, kv_rank=4 * hd, scale=hd ** -0.5)
        kinds = [{"type": "parallel", "mixer": parallel}, {"type": "latent_attention", "mixer": rows},
                 {"type": "channel_delta", "mixer": delta}, {"type": "channel_delta", "mixer": delta}]
        built = [dict(kinds[i % 4], mlp=moe) for i in range(layers)]
        for i in range(5, layers, 4):  # the later latent layers read the first one's rows
            built[i] = dict(built[i], mixer=dict(rows, kv_from=1))
        return dict(out, embedding={"bigram": {"buckets": 65521, "mul_prev": 31, "mul_cur": 7}}, layers=built)
    if case["design"] == "zikezen":  # `layers` layer runs: the second and third layer run twice
        mixer = {"left": dict(softmax, mask={"size": 2048}, rot={"base": 1e6, "dims": hd // 2, "scaling": {
                     "factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}),
                 "right": dict(base, tau=16.0, decay_rank=hd // 2), "left_scale": 0.7, "right_scale": 0.7}
        moe = {"kind": "moe", "expert": {"ff": narrow}, "router": {"experts": 32, "top": 4}}
        return dict(out, max_positions=32768, embedding={"scale": 1.0}, token_side={"dim": 64}, logit_softcap=30.0,
                    loop={"start": 1, "stop": 3, "times": 2},
                    layers=[{"type": "parallel", "mixer": mixer, "mlp": moe if i % 2 else dense} for i in range(layers - 2)])
    if case["design"] == "getodra":
        fixed = dict(base, decay=[1.0 - 0.4 * 2.0 ** (-11.0 * h / (heads - 1)) for h in range(heads)])
        rows = dict(latent, rot={"base": 1e6, "dims": hd // 2, "scaling": dict(stretched, fast=32.0, slow=1.0)})
        built = [{"type": "latent_attention", "mixer": rows, "mlp": dense} if i % 2
                 else {"type": "lightning", "mixer": fixed, "mlp": dense} for i in range(layers)]
        built[5] = dict(built[5], weights_of=3)
        return dict(out, max_positions=32768, canon={"taps": 4}, layers=built)
    if case["design"] == "mulenex":
        attention = {"type": "attention", "mixer": dict(softmax, softcap=50.0, v_mix=True, q_temp={"coef": 0.1, "every": 8192})}
        memory = {"type": "mlstm", "mixer": dict(base, gate_cap=15.0)}
        moe = {"kind": "moe", "expert": {"ff": narrow}, "router": {"experts": 32, "top": 3}, "shared": {"ff": narrow}}
        return dict(out, layers=[dict(memory if i % 2 else attention, mlp=(dense, moe, moe, dense)[i % 4])
                                 for i in range(layers)])
    raise ValueError(case["design"])


def layer_runs(cfg):
    """(layer, the layer whose tensors it uses, does the embedding's output join before it) in order of running."""
    if "num_hidden_layers" in cfg:
        return [(i, i, False) for i in range(cfg["num_hidden_layers"])]
    layers, loop = cfg["layers"], cfg.get("loop")
    own = [layer.get("weights_of", i) for i, layer in enumerate(layers)]
    order = [(i, False) for i in range(len(layers))]
    if loop:
        a, b = loop["start"], loop["stop"]
        order = order[:b] + [(i, i == a) for i in range(a, b)] * (loop["times"] - 1) + order[b:]
    return [(i, own[i], joins) for i, joins in order]


# What a trained checkpoint's tensors look like, by the end of the tensor's name: (how, first number, second).  As in
# trained models a branch adds a small part of the stream it reads: the last products of the branches are
# narrow, and so are the weights of norms behind a branch.  "fan in": about zero, the second number over the root of the inputs.
SPREADS = {
    "embed": ("normal", 0.0, 0.3), "embed_tokens.weight": ("normal", 0.0, 0.3), "bigram": ("normal", 0.0, 0.1),
    "pos": ("normal", 0.0, 0.1), "side.embed": ("normal", 0.0, 0.5), ".sink": ("normal", 0.0, 1.0),
    ".A_log": ("log of uniform", 1.0, 16.0), ".dt_bias": ("inverse softplus", 1e-3, 1e-1), ".conv": ("normal", 0.0, 0.3),
    ".f.b": ("uniform", 2.0, 6.0), "a2.b": ("normal", 1.0, 1.0), ".correction": ("normal", 0.0, 0.005),
    "router": ("fan in", 0.0, 4.0), ".in": ("normal", 0.25, 0.05), ".out": ("normal", 1.0, 0.1),
    ".hc1.mix": ("identity", 0.0, 0.05), ".hc2.mix": ("identity", 0.0, 0.05), "vmix": ("uniform", 0.2, 0.6),
    "canon1": ("normal", 0.0, 0.1), "canon2": ("normal", 0.0, 0.1), "q_proj.weight": ("fan in", 0.0, 1.2),
    "k_proj.weight": ("fan in", 0.0, 1.2), "o_proj.weight": ("fan in", 0.0, 0.2), "down_proj.weight": ("fan in", 0.0, 0.2),
    ".o": ("fan in", 0.0, 0.2), ".down": ("fan in", 0.0, 0.2), "norm": ("normal", 1.0, 0.1), "norm1": ("normal", 1.0, 0.1),
    "norm2": ("normal", 1.0, 0.1), "norm1b": ("normal", 0.1, 0.01), "norm2b": ("normal", 0.05, 0.005),
    "side.norm": ("normal", 0.05, 0.005), "ls1": ("normal", 1.0, 0.1), "ls2": ("normal", 1.0, 0.1),
    "layernorm.weight": ("normal", 1.0, 0.1), "norm.weight": ("normal", 1.0, 0.1), ".b": ("normal", 0.0, 0.02),
    ".bias": ("normal", 0.0, 0.02),
}
# norms whose weights are stored less one, and norms behind a branch that the names above do not tell
OFFSET_NORMS = {"dagavik": ("norm1", "norm2", "final.norm"), "mulenex": ("norm1", "norm1b", "norm2", "norm2b", "final.norm")}
BRANCH_NORMS = {"danonex": ("norm1", "norm2"), "getodra": ("norm1", "norm2")}


def draw_tensor(case, seed, name, shape):
    """The tensor `name` of the case's model, from the seed and the name alone."""
    device = "cuda:0"
    gen = torch.Generator(device=device).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
    ending = max((e for e in SPREADS if name.endswith(e)), key=len, default=None)
    how, a, b = SPREADS[ending] if ending else ("fan in", 0.0, 0.8)
    if how == "fan in":
        how, b = "normal", b / math.sqrt(shape[-1])
    if ".mlp.e" in name and name.endswith(".down"):
        b = 0.1 * b  # a token's experts add up, and a close choice among them may fall either way
    if name.endswith(BRANCH_NORMS.get(case["design"], "-")):
        a, b = 0.2 * a, 0.2 * b
    if name.endswith(OFFSET_NORMS.get(case["design"], "-")):
        a -= 1.0
    if how in ("normal", "identity"):
        out = torch.randn(shape, generator=gen, device=device).mul_(b).add_(a)
        if how == "identity":
            out += torch.eye(shape[0], device=device)
    else:
        u = torch.rand(shape, generator=gen, device=device)
        if how == "uniform":
            out = a + (b - a) * u
        elif how == "log of uniform":
            out = torch.log(a + (b - a) * u)
        else:  # the number whose softplus is spread evenly over the logarithm from a to b
            out = torch.log(torch.expm1(torch.exp(math.log(a) + (math.log(b) - math.log(a)) * u)))
    return out.to(getattr(torch, case["dtype"]))


class Drawn(Mapping):
    """name -> tensor, drawn when it is looked up, so that no weight lies in memory twice."""

    def __init__(self, case, seed, shapes):
        self.case, self.seed, self.shapes = case, seed, shapes

    def __getitem__(self, name):
        return draw_tensor(self.case, self.seed, name, tuple(self.shapes[name]))

    def __contains__(self, name):
        return name in self.shapes

    def __iter__(self):
        return iter(self.shapes)

    def __len__(self):
        return len(self.shapes)


def prepare(case, seed):
    """The model, its cache, a step runner, the sequences' tokens; for kind "step" the contexts in the cache."""
    import paged_attention_engine_amd as pae

    config = pae.read_config_dict(config_of(case))
    plan = config.plan()
    model = pae.Model(plan, getattr(torch, case["dtype"]), "cuda:0")
    model.bind(Drawn(case, seed, pae.expected_tensors(plan)))
    sequences, tokens = sequences_of(case), tokens_of(case, seed)
    pages = sum(-(-len(t) // BLOCK) + 1 for t in tokens)
    cache = model.new_cache(BLOCK, pages, len(sequences))
    runner = pae.StepRunner(model, cache)
    state = {"case": case, "cache": cache, "runner": runner, "entry": pae.StepEntry, "sequences": sequences,
             "tokens": [tuple(t) for t in tokens]}
    if case["kind"] == "step":
        batch, room = [], CHUNK
        for s, (held, new) in enumerate(sequences):
            cache.create_sequence(s)
            done = 0
            while done < held:
                part = min(room, held - done)
                cache.reserve(s, part)
                batch.append(pae.StepEntry(s, state["tokens"][s][done:done + part]))
                done, room = done + part, room - part
                if room == 0 or done < held:
                    runner.run(batch)
                    batch, room = [], CHUNK
        if batch:
            runner.run(batch)
        for s, (held, new) in enumerate(sequences):
            cache.reserve(s, new)
        state["step"] = [pae.StepEntry(s, state["tokens"][s][held:held + new], (new - 1,))
                         for s, (held, new) in enumerate(sequences)]
    return state


def run(state):
    """One pass: the logits of every sequence's last token of the first step, then of every later step."""
    cache, runner, entry = state["cache"], state["runner"], state["entry"]
    if state["case"]["kind"] == "step":
        return [runner.run(state["step"])]
    sequences, tokens, steps = state["sequences"], state["tokens"], state["case"]["steps"]
    first = []
    for s, (_, new) in enumerate(sequences):
        cache.create_sequence(s)
        cache.reserve(s, new)
        first.append(entry(s, tokens[s][:new], (new - 1,)))
    out = [runner.run(first)]
    for k in range(steps):
        for s in range(len(sequences)):
            cache.release_passed(s)
            cache.reserve(s, 1)
        logits = runner.run([entry(s, (tokens[s][new + k],), (0,)) for s, (_, new) in enumerate(sequences)])
        out.append(logits.clone())  # the runner may write the next step's logits over these
    for s in range(len(sequences)):
        cache.free_sequence(s)
    return out


# --------------------------------------------------------------------------- what a pass cannot do without


def work(case):
    """Bytes: every weight that a step uses, the cache and state that it reads and writes, the logits.  FLOPs:
    two per weight and token, and per key that a query sees two per number of the key and of the value."""
    cfg, elem = config_of(case), 2 if case["dtype"] == "bfloat16" else 4
    hidden, _, heads, kv, hd, ff, _ = SIZES[case["size"]]
    vocab, sequences = VOCAB[case["size"]], sequences_of(case)
    steps = [sequences] + [[(held + new + k, 1) for held, new in sequences] for k in range(case["steps"])]
    flops = moved = 0.0
    for step in steps:
        T, S = sum(new for _, new in step), len(step)
        flops += 2.0 * S * vocab * hidden
        moved += vocab * hidden * elem + S * vocab * 4 + T * hidden * elem
        seen = set()
        for i, own, _ in layer_runs(cfg):
            layer = cfg["layers"][i] if "layers" in cfg else {"type": "qwen2", "mixer": {}, "mlp": {"kind": "dense"}}
            mlp, new_weights = layer["mlp"], own not in seen
            seen.add(own)
            gated = case["design"] in ("qwen2", "ritalorn", "zikezen", "getodra") or mlp["kind"] == "moe"
            if mlp["kind"] == "dense":
                n = (3 if gated else 2) * hidden * ff
                flops, moved = flops + 2.0 * T * n, moved + n * elem * new_weights
            else:
                n, top, count = 3 * hidden * mlp["expert"]["ff"], mlp["router"]["top"], mlp["router"]["experts"]
                used = count * (1.0 - (1.0 - top / count) ** T)
                if mlp.get("shared"):
                    flops, moved = flops + 2.0 * T * n, moved + n * elem * new_weights
                flops, moved = flops + 2.0 * T * top * n, moved + used * n * elem * new_weights
            for kind, m in mixers_of(layer):
                weights, width, kept = mixer_sizes(kind, m, hidden, heads, kv, hd)
                flops, moved = flops + 2.0 * T * weights, moved + weights * elem * new_weights
                window = (m.get("mask") or {}).get("size") or 1 << 30
                for held, new in step:
                    if kind in ("softmax", "latent"):
                        if m.get("mask") and layer["type"] == "attention":  # chunks: a query sees its own chunk's keys
                            pairs = sum(p % window + 1 for p in range(held, held + new))
                        else:
                            pairs = sum(min(p + 1, window) for p in range(held, held + new))
                        flops += 2.0 * heads * width * pairs
                        moved += kept * elem * (min(held + new, window + new))
                    else:  # a state of heads x hd x hd numbers in 32 bits, read, changed and read again
                        flops += 6.0 * heads * hd * hd * new
                        moved += 8.0 * heads * hd * hd
    return {"bytes": moved, "flops": flops}


def mixers_of(layer):
    """[(softmax | latent | recurrent, config)] of a layer's mixers."""
    kind, m = layer["type"], layer["mixer"]
    if kind == "parallel":
        return [("softmax", m["left"]), ("recurrent", m["right"])]
    if kind in ("qwen2", "attention"):
        return [("softmax", m)]
    return [("latent" if kind == "latent_attention" else "recurrent", m)]


def mixer_sizes(kind, m, hidden, heads, kv, hd):
    """(weights, numbers of a key and a value, numbers cached per token) of a mixer."""
    if kind == "softmax":
        return 2 * (heads + kv) * hd * hidden, 2 * hd, 2 * kv * hd
    if kind == "latent":
        R = m.get("rot_dim", 0)
        up = 2 * heads * hd * m["kv_rank"]
        return hidden * (heads * (hd + R) + m["kv_rank"] + R + heads * hd) + up, 2 * hd + R, m["kv_rank"] + R
    groups = m.get("kv_heads", heads)
    return hidden * hd * (2 * groups + 3 * heads), 0, 0


def tolerance(case):
    """Two correct implementations differ by the rounding of what they store.  Measured against 64 bits (relative error of
    the logits): bfloat16 0.004 to 0.009; where a token's experts are chosen by scores that nearly tie, rounding
    chooses others, and single rows are up to 0.02 off; float32 1.0e-6 to 2.5e-6.  Four times that, and `max`
    (of single logits, over the root mean square of all) for the rows whose experts changed."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.6}


# --------------------------------------------------------------------------- the same in 64 bits
# Whole sequences, no cache: the tokens of all sequences lie one after another in `x`, products run over all of
# them, and what looks along a sequence runs sequence by sequence.


def over_rms(x, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def silu(z):
    return z * torch.sigmoid(z)


def gelu_tanh(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def soft_cap(z, cap):
    return cap * torch.tanh(z / cap) if cap else z


def pair_frequencies(rot):
    """(frequency of every rotated pair, multiplier of the cosines and sines); `scaling` stretches the slow ones, by a
    ramp over the pairs (fast, slow) or by their wavelength (low, high)."""
    dims, scaling = rot["dims"], rot.get("scaling")
    i = torch.arange(dims // 2, dtype=torch.float64, device="cuda:0")
    f = float(rot["base"]) ** (-2.0 * i / dims)
    if not scaling:
        return f, 1.0
    factor, original = scaling["factor"], scaling["original"]
    if "low" in scaling:
        wave, low, high = 2.0 * math.pi / f, scaling["low"], scaling["high"]
        keep = torch.clamp((original / wave - low) / (high - low), 0.0, 1.0)
        return f / factor * (1.0 - keep) + f * keep, 1.0
    place = [dims * math.log(original / (2.0 * math.pi * scaling[k])) / (2.0 * math.log(rot["base"])) for k in ("fast", "slow")]
    low, high = max(math.floor(place[0]), 0), min(math.ceil(place[1]), dims - 1)
    ramp = torch.clamp((i - low) / max(high - low, 0.001), 0.0, 1.0)
    return f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0


def rotate(x, positions, rot, halves):
    """x [T, heads, dim]: the first rot.dims features turn, feature i with i + dims/2 (`halves`) or 2i with 2i + 1."""
    if not rot or not rot.get("dims"):
        return x
    f, multiplier = pair_frequencies(rot)
    angle = positions.double()[:, None, None] * f
    c, s, dims, out = torch.cos(angle) * multiplier, torch.sin(angle) * multiplier, rot["dims"], x.clone()
    first, second = (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
    u, v = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * c - v * s, v * c + u * s
    return out


def attend(q, k, v, scale, spans, cap=None, window=None, chunk=None, sink=None, slopes=None):
    """Softmax attention, sequence by sequence: q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H, V].  `sink` [H]: the score
    of a key without a value; `slopes` [H]: taken off a score per token of distance."""
    H, G, out = q.shape[1], k.shape[1], torch.empty((q.shape[0], q.shape[1], v.shape[2]), dtype=q.dtype, device=q.device)
    for a, n in spans:
        kk = k[a:a + n].repeat_interleave(H // G, 1).permute(1, 2, 0)
        vv = v[a:a + n].repeat_interleave(H // G, 1).permute(1, 0, 2).contiguous()
        place = torch.arange(n, device=q.device)
        unit = max(1, min(n, (1 << 27) // (H * n)))
        for at in range(0, n, unit):
            here = place[at:at + unit, None]
            s = soft_cap(torch.matmul(q[a + at:a + min(n, at + unit)].permute(1, 0, 2).contiguous(), kk.contiguous()) * scale, cap)
            if slopes is not None:
                s = s - slopes[:, None, None] * (here - place).double()
            hidden = place > here
            if window:
                hidden = hidden | (here - place >= window)
            if chunk:
                hidden = hidden | (here // chunk != place // chunk)
            s = s.masked_fill(hidden, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[:, None, None].expand(-1, s.shape[1], 1)], -1)
            p = torch.softmax(s, -1)[..., :n]
            out[a + at:a + at + p.shape[1]] = torch.matmul(p, vv).permute(1, 0, 2)
    return out


def along(x, spans, taps, keep):
    """Causal convolution of every channel (taps [C, n], the last column meets the current token), sequence by
    sequence; `keep`: the input itself is added."""
    out = x.clone() if keep else torch.zeros_like(x)
    for a, n in spans:
        for b in range(min(taps.shape[1], n)):
            out[a + b:a + n] += taps[:, taps.shape[1] - 1 - b] * x[a:a + n - b]
    return out


def recurrence(q, k, v, decay, spans, beta=None):
    """State S [H, D, V] per sequence: S <- decay S (per row);  u = v, or beta (v - S^T k);  S <- S + k u^T;  o = S^T q."""
    out = torch.empty_like(v)
    for a, n in spans:
        S = torch.zeros((v.shape[1], q.shape[2], v.shape[2]), dtype=v.dtype, device=v.device)
        for t in range(a, a + n):
            S = S * decay[t][:, :, None]
            u = v[t] if beta is None else beta[t][:, None] * (v[t] - torch.einsum("hdv,hd->hv", S, k[t]))
            S = torch.baddbmm(S, k[t][:, :, None], u[:, None, :])
            out[t] = torch.bmm(q[t][:, None, :], S)[:, 0]
    return out


def memory(q, k, v, log_in, log_keep, spans):
    """Matrix memory with exponential gates: S <- keep S + take k v^T, n likewise, in units of exp(m), m the running
    maximum; read out over max(|n q|, exp(-m)) + 1e-6."""
    out = torch.empty_like(v)
    v1 = torch.cat([v, torch.ones_like(v[..., :1])], -1)
    for a, n in spans:
        S = torch.zeros((q.shape[1], q.shape[2], v1.shape[2]), dtype=v.dtype, device=v.device)
        m = torch.zeros(q.shape[1], dtype=v.dtype, device=v.device)
        for t in range(a, a + n):
            old, m = log_keep[t] + m, torch.maximum(log_keep[t] + m, log_in[t])
            S = torch.baddbmm(S * torch.exp(old - m)[:, None, None], (k[t] * torch.exp(log_in[t] - m)[:, None])[:, :, None], v1[t][:, None, :])
            o = torch.bmm(q[t][:, None, :], S)[:, 0]
            out[t] = o[:, :-1] / (torch.maximum(o[:, -1].abs(), torch.exp(-m)) + 1e-6)[:, None]
    return out


class Exact:
    def __init__(self, case, seed):
        self.case, self.seed, self.cfg = case, seed, config_of(case)
        self.hidden, _, self.H, self.G, self.D, self.ff, self.tied = SIZES[case["size"]]
        self.eps = 1e-6
        tokens = tokens_of(case, seed)
        lengths = [len(t) for t in tokens]
        starts = [sum(lengths[:i]) for i in range(len(lengths))]
        self.spans = list(zip(starts, lengths))
        self.ids = torch.tensor([t for seq in tokens for t in seq], device="cuda:0")
        self.place = torch.cat([torch.arange(n, device="cuda:0") for n in lengths])
        first = [start + held + new - 1 for start, (held, new) in zip(starts, sequences_of(case))]
        self.wanted = [torch.tensor(first, device="cuda:0") + k for k in range(case["steps"] + 1)]

    def w(self, name, *shape):
        return draw_tensor(self.case, self.seed, name, shape).double()

    def rows(self, name, count, width, ids):
        return draw_tensor(self.case, self.seed, name, (count, width))[ids].double()

    def times(self, x, name, rows, bias=None):
        y = x @ self.w(name, rows, x.shape[-1]).T
        return y if bias is None else y + self.w(bias, rows)

    def logits(self, x, name):
        picked = [x[rows] for rows in self.wanted]
        weight = draw_tensor(self.case, self.seed, name, (VOCAB[self.case["size"]], self.hidden))
        flat, part = torch.cat(picked), 16384
        y = torch.cat([flat @ weight[i:i + part].double().T for i in range(0, weight.shape[0], part)], -1)
        return list(y.split([p.shape[0] for p in picked]))

    def heads(self, x, dim):
        return x.view(x.shape[0], -1, dim)

    def sizes(self, m):
        return m["heads"] * m["dim"], m.get("kv_heads", m["heads"]) * m["dim"], m["dim"]

    def experts(self, p, mlp, h, chosen, weights):
        out, ff = torch.zeros_like(h), mlp["expert"]["ff"]
        for e in range(mlp["router"]["experts"]):
            t, slot = (chosen == e).nonzero(as_tuple=True)
            if len(t):
                out.index_add_(0, t, weights[t, slot][:, None] * self.gated(h[t], f"{p}e{e}.", ff, silu))
        return out

    def gated(self, h, p, ff, act):
        return self.times(act(self.times(h, p + "gate", ff)) * self.times(h, p + "up", ff), p + "down", self.hidden)

    # one method per design: x -> the final stream's logits
    def qwen2(self):
        H, G, D, hidden = self.H, self.G, self.D, self.hidden
        vocab, eps, rot = VOCAB[self.case["size"]], self.eps, {"base": 1e6, "dims": D}
        x = self.rows("model.embed_tokens.weight", vocab, hidden, self.ids)
        for i in range(self.case["layers"]):
            p = f"model.layers.{i}."
            h = over_rms(x, eps) * self.w(p + "input_layernorm.weight", hidden)
            q, k, v = (self.heads(self.times(h, f"{p}self_attn.{n}_proj.weight", rows * D, f"{p}self_attn.{n}_proj.bias"), D)
                       for n, rows in (("q", H), ("k", G), ("v", G)))
            q, k = rotate(q, self.place, rot, True), rotate(k, self.place, rot, True)
            o = attend(q, k, v, D ** -0.5, self.spans)
            x = x + self.times(o.reshape(x.shape[0], H * D), p + "self_attn.o_proj.weight", hidden)
            h = over_rms(x, eps) * self.w(p + "post_attention_layernorm.weight", hidden)
            act = silu(self.times(h, p + "mlp.gate_proj.weight", self.ff)) * self.times(h, p + "mlp.up_proj.weight", self.ff)
            x = x + self.times(act, p + "mlp.down_proj.weight", hidden)
        return self.logits(over_rms(x, eps) * self.w("model.norm.weight", hidden),
                           "model.embed_tokens.weight" if self.tied else "lm_head.weight")

    def delta(self, h, p, m):
        Q, K, D = self.sizes(m)
        per = m["heads"] // m["kv_heads"]
        conv = lambda n, rows: self.heads(silu(along(self.times(h, p + n, rows), self.spans, self.w(f"{p}{n}.conv", rows, m["conv"]), False)), D)
        unit = lambda z: z / torch.sqrt(z.pow(2).sum(-1, keepdim=True) + 1e-6)
        q, k, v = unit(conv("q", K)) * D ** -0.5, unit(conv("k", K)), conv("v", Q)
        beta, rate = torch.sigmoid(self.times(h, p + "b", m["heads"])), torch.exp(self.w(p + "A_log", m["heads"]))
        if "decay_rank" in m:
            step = self.heads(self.times(self.times(h, p + "a1", m["decay_rank"]), p + "a2", Q) + self.w(p + "dt_bias", Q), D)
            gate = torch.sigmoid(self.times(self.times(h, p + "g1", m["gate_rank"]), p + "g2", Q))
        else:
            step = (self.times(h, p + "a", m["heads"]) + self.w(p + "dt_bias", m["heads"]))[..., None]
            gate = silu(self.times(h, p + "g", Q))
        decay = torch.exp(-rate[:, None] * torch.nn.functional.softplus(step)).expand(-1, -1, D)
        o = recurrence(q.repeat_interleave(per, 1), k.repeat_interleave(per, 1), v, decay, self.spans, beta)
        o = over_rms(o, self.eps) * self.w(p + "norm", D) * self.heads(gate, D)
        return self.times(o.reshape(h.shape[0], Q), p + "o", self.hidden)

    def danonex(self):
        hidden, eps = self.hidden, self.eps
        x = self.rows("embed", self.cfg["vocab"], hidden, self.ids)
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            if layer["type"] == "delta":
                y = self.delta(x, p + "mix.", m)
            else:
                Q, K, D = self.sizes(m)
                q = self.heads(over_rms(self.times(x, p + "mix.q", Q), eps) * self.w(p + "mix.q.norm", Q), D)
                k = self.heads(over_rms(self.times(x, p + "mix.k", K), eps) * self.w(p + "mix.k.norm", K), D)
                v = self.heads(self.times(x, p + "mix.v", K), D)
                q, k = rotate(q, self.place, m["rot"], False), rotate(k, self.place, m["rot"], False)
                o = attend(q, k, v, m["scale"], self.spans, cap=m["softcap"], sink=self.w(p + "mix.sink", m["heads"]))
                y = self.times(o.reshape(x.shape[0], Q), p + "mix.o", hidden)
            x = x + 0.5 * over_rms(y, eps) * self.w(p + "norm1", hidden)
            up = torch.nn.functional.gelu(self.times(x, p + "mlp.up", self.ff))
            x = x + 0.5 * over_rms(self.times(up, p + "mlp.down", hidden), eps) * self.w(p + "norm2", hidden)
        return [0.5 * y for y in self.logits(over_rms(x, eps) * self.w("final.norm", hidden), "embed")]

    def latent(self, h, p, m, halves, rows=None):
        """Latent attention up to the heads' outputs, and the rows (latent, rotated part) it read."""
        Q, _, D = self.sizes(m)
        C, R, H = m["kv_rank"], m.get("rot_dim", 0), m["heads"]
        q = self.heads(self.times(h, p + "q", H * (D + R)), D + R)
        if rows is None:
            down = self.times(h, p + "dkv", C + R)
            rows = (over_rms(down[:, :C], self.eps) * self.w(p + "dkv.norm", C), rotate(down[:, None, C:], self.place, m.get("rot"), halves))
        c, turned = rows
        k = torch.cat([self.heads(self.times(c, p + "uk", Q), D), turned.expand(-1, H, -1)], -1)
        q = torch.cat([q[..., :D], rotate(q[..., D:], self.place, m.get("rot"), halves)], -1)
        sink = self.w(p + "sink", H) if self.case["design"] == "dagavik" else None
        o = attend(q, k, self.heads(self.times(c, p + "uv", Q), D), m["scale"], self.spans,
                   window=(m.get("mask") or {}).get("size"), sink=sink)
        return o, rows

    def ritalorn(self):
        hidden, eps, S = self.hidden, self.eps, self.cfg["streams"]
        X = self.rows("embed", self.cfg["vocab"], hidden, self.ids)[None].expand(S, -1, -1)
        kept = {}
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            Q, K, D = self.sizes(m)

            def mixer(h):
                if layer["type"] == "latent_attention":
                    o, _ = self.latent(h, p + "mix.", m, False)
                    return self.times(o.reshape(h.shape[0], Q), p + "mix.o", hidden)
                conv = lambda n, rows: self.heads(along(self.times(h, f"{p}mix.{n}", rows, f"{p}mix.{n}.b"), self.spans,
                                                        self.w(f"{p}mix.{n}.conv", rows, m["conv"]), False), D)
                source = m.get("kv_from", i)
                if source == i:
                    kept[i] = over_rms(conv("k", K), eps), conv("v", K)
                slopes = torch.tensor([2.0 ** (-8.0 * (j + 1) / m["heads"]) for j in range(m["heads"])], dtype=torch.float64, device="cuda:0")
                o = attend(over_rms(conv("q", Q), eps), *kept[source], m["scale"], self.spans, chunk=m["mask"]["size"], slopes=slopes)
                o = o.reshape(h.shape[0], Q) * torch.sigmoid(self.times(h, p + "mix.g", Q))
                return self.times(o, p + "mix.o", hidden, p + "mix.o.b")

            for n, sublayer in (("1", mixer), ("2", lambda h: self.gated(h, p + "mlp.", self.ff, gelu_tanh))):
                u = torch.einsum("s,stw->tw", self.w(f"{p}hc{n}.in", S), X)
                y = self.w(f"{p}ls{n}", hidden) * sublayer(over_rms(u, eps) * self.w(f"{p}norm{n}", hidden))
                X = torch.einsum("st,snw->tnw", self.w(f"{p}hc{n}.mix", S, S), X) + self.w(f"{p}hc{n}.out", S)[:, None, None] * y
        return [soft_cap(y, self.cfg["logit_softcap"])
                for y in self.logits(over_rms(X.sum(0), eps) * self.w("final.norm", hidden), "head")]

    def matrix_memory(self, h, p, m):
        Q, _, D = self.sizes(m)
        q, k, v = self.heads(self.times(h, p + "q", Q), D) * D ** -0.5, self.heads(self.times(h, p + "k", Q), D), self.heads(self.times(h, p + "v", Q), D)
        log_in = soft_cap(self.times(h, p + "i", m["heads"], p + "i.b"), m["gate_cap"])
        log_keep = torch.nn.functional.logsigmoid(soft_cap(self.times(h, p + "f", m["heads"], p + "f.b"), m["gate_cap"]))
        o = over_rms(memory(q, k, v, log_in, log_keep, self.spans), self.eps).reshape(h.shape[0], Q)
        return self.times(o * self.w(p + "norm", Q) * torch.sigmoid(self.times(h, p + "g", Q)), p + "o", self.hidden)

    def dagavik(self):
        hidden, eps, cfg = self.hidden, self.eps, self.cfg
        x = self.rows("embed", cfg["vocab"], hidden, self.ids)
        pairs, before = cfg["embedding"]["bigram"], torch.roll(self.ids, 1)
        row = torch.where(self.place == 0, pairs["buckets"], (before * pairs["mul_prev"] + self.ids * pairs["mul_cur"]) % pairs["buckets"])
        x = x + self.rows("bigram", pairs["buckets"] + 1, hidden, row)
        rows = {}
        for i, layer in enumerate(cfg["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = over_rms(x, eps) * (1.0 + self.w(p + "norm1", hidden))
            if layer["type"] == "parallel":
                left = m["left"]
                Q, K, D = self.sizes(left)
                q, k, v = (self.heads(self.times(h, f"{p}mix.left.{n}", r, f"{p}mix.left.{n}.b"), D) for n, r in (("q", Q), ("k", K), ("v", K)))
                q, k = rotate(q, self.place, left["rot"], True), rotate(k, self.place, left["rot"], True)
                o = attend(q, k, v, left["scale"], self.spans, window=left["mask"]["size"])
                y = (m["left_scale"] * self.times(o.reshape(x.shape[0], Q), p + "mix.left.o", hidden)
                     + m["right_scale"] * self.matrix_memory(h, p + "mix.right.", m["right"]))
            elif layer["type"] == "latent_attention":
                o, read = self.latent(h, p + "mix.", m, True, rows.get(m.get("kv_from")))
                rows[i] = read
                y = self.times(o.reshape(x.shape[0], -1), p + "mix.o", hidden)
            else:
                y = self.delta(h, p + "mix.", m)
            h = over_rms(x, eps) * (1.0 + self.w(p + "norm2", hidden))
            r = mlp["router"]
            s, groups = torch.softmax(self.times(h, p + "mlp.router", r["experts"]), -1), r["groups"]
            best = s.view(-1, groups["count"], r["experts"] // groups["count"]).amax(-1).topk(groups["keep"], -1).indices
            allowed = torch.zeros((s.shape[0], groups["count"]), dtype=torch.bool, device=s.device).scatter_(1, best, True)
            chosen = s.masked_fill(~allowed.repeat_interleave(r["experts"] // groups["count"], 1), -1.0).topk(r["top"], -1).indices
            x = x + y + self.experts(p + "mlp.", mlp, h, chosen, s.gather(1, chosen) * r["scale"])
        return self.logits(over_rms(x, eps) * (1.0 + self.w("final.norm", hidden)), "head")

    def zikezen(self):
        hidden, eps, cfg = self.hidden, self.eps, self.cfg
        x = self.rows("embed", cfg["vocab"], hidden, self.ids) + self.rows("pos", cfg["max_positions"], hidden, self.place)
        start, side, count = x, cfg["token_side"]["dim"], len(cfg["layers"])
        table = self.rows("side.embed", cfg["vocab"], count * side, self.ids)
        for i, _, joins in layer_runs(cfg):
            p, m, mlp = f"l{i}.", cfg["layers"][i]["mixer"], cfg["layers"][i]["mlp"]
            x = x + start if joins else x
            h = over_rms(x, eps) * self.w(p + "norm1", hidden)
            left, right = m["left"], m["right"]
            Q, K, D = self.sizes(left)
            q, k, v = (self.heads(self.times(h, f"{p}mix.left.{n}", r, f"{p}mix.left.{n}.b"), D) for n, r in (("q", Q), ("k", K), ("v", K)))
            q = rotate(over_rms(q, eps) * self.w(p + "mix.left.q.norm", D), self.place, left["rot"], False)
            k = rotate(over_rms(k, eps) * self.w(p + "mix.left.k.norm", D), self.place, left["rot"], False)
            o = attend(q, k, v, left["scale"], self.spans, window=left["mask"]["size"],
                       sink=torch.zeros(left["heads"], dtype=torch.float64, device="cuda:0"))
            y = m["left_scale"] * self.times(o.reshape(x.shape[0], Q), p + "mix.left.o", hidden)
            at = p + "mix.right."
            Q, _, D = self.sizes(right)
            q, k, v = (self.heads(self.times(h, at + n, Q), D) for n in "qkv")
            z = self.times(self.times(h, at + "a1", right["decay_rank"]), at + "a2", Q, at + "a2.b")
            decay = self.heads(torch.exp(torch.nn.functional.logsigmoid(z) / right["tau"]), D)
            o = over_rms(recurrence(q * D ** -0.5, k, v, decay, self.spans), eps) * self.w(at + "norm", D)
            o = o.reshape(x.shape[0], Q) * silu(self.times(h, at + "g", Q))
            y = y + m["right_scale"] * self.times(o, at + "o", hidden)
            x = x + over_rms(y, eps) * self.w(p + "norm1b", hidden)
            h = over_rms(x, eps) * self.w(p + "norm2", hidden)
            if mlp["kind"] == "dense":
                y = self.gated(h, p + "mlp.", self.ff, silu)
            else:
                r = mlp["router"]
                s = torch.softmax(self.times(h, p + "mlp.router", r["experts"]), -1)
                chosen = (s + self.w(p + "mlp.correction", r["experts"])).topk(r["top"], -1).indices
                y = self.experts(p + "mlp.", mlp, h, chosen, s.gather(1, chosen))
            x = x + over_rms(y, eps) * self.w(p + "norm2b", hidden)
            g = gelu_tanh(self.times(x, p + "side.gate", side)) * table[:, i * side:(i + 1) * side]
            x = x + over_rms(self.times(g, p + "side.proj", hidden), eps) * self.w(p + "side.norm", hidden)
        return [soft_cap(y, cfg["logit_softcap"]) for y in self.logits(over_rms(x, eps) * self.w("final.norm", hidden), "head")]

    def getodra(self):
        hidden, eps, cfg, taps = self.hidden, self.eps, self.cfg, self.cfg["canon"]["taps"]
        x = self.rows("embed", cfg["vocab"], hidden, self.ids) + self.rows("pos", cfg["max_positions"], hidden, self.place)
        for i, own, _ in layer_runs(cfg):
            p, m = f"l{own}.", cfg["layers"][i]["mixer"]
            Q, _, D = self.sizes(m)
            h = along(x, self.spans, self.w(p + "canon1", hidden, taps), True)
            if cfg["layers"][i]["type"] == "lightning":
                q, k, v = (self.heads(silu(self.times(h, f"{p}mix.{n}", Q)), D) for n in "qkv")
                decay = torch.tensor(m["decay"], dtype=torch.float64, device="cuda:0")[None, :, None].expand(x.shape[0], -1, D)
                o = over_rms(recurrence(q, k, v, decay, self.spans).reshape(x.shape[0], Q), eps) * self.w(p + "mix.norm", Q)
                o = o * torch.sigmoid(self.times(h, p + "mix.g", Q))
            else:
                o, _ = self.latent(h, p + "mix.", m, True)
                o = (o * torch.sigmoid(self.times(h, p + "mix.g", m["heads"]))[..., None]).reshape(x.shape[0], Q)
            x = x + over_rms(self.times(o, p + "mix.o", hidden), eps) * self.w(p + "norm1")
            h = along(x, self.spans, self.w(p + "canon2", hidden, taps), True)
            x = x + over_rms(self.gated(h, p + "mlp.", self.ff, gelu_tanh), eps) * self.w(p + "norm2")
        return self.logits(over_rms(x, eps) * self.w("final.norm"), "head")

    def mulenex(self):
        hidden, eps, cfg = self.hidden, self.eps, self.cfg
        turn = 10000.0 ** (-2.0 * torch.arange(hidden // 2, dtype=torch.float64, device="cuda:0") / hidden) * self.place.double()[:, None]
        x = self.rows("embed", cfg["vocab"], hidden, self.ids) + torch.stack([torch.sin(turn), torch.cos(turn)], -1).reshape(-1, hidden)
        norm = lambda name, y: over_rms(y, eps) * (1.0 + self.w(name, hidden))
        values = None
        for i, layer in enumerate(cfg["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = norm(p + "norm1", x)
            if layer["type"] == "mlstm":
                y = self.matrix_memory(h, p + "mix.", m)
            else:
                Q, K, D = self.sizes(m)
                temperature = 1.0 + m["q_temp"]["coef"] * torch.log((self.place + 1) // m["q_temp"]["every"] + 1.0).double()
                q = over_rms(self.heads(self.times(h, p + "mix.q", Q), D), eps) * self.w(p + "mix.q.norm", D) * temperature[:, None, None]
                k = over_rms(self.heads(self.times(h, p + "mix.k", K), D), eps) * self.w(p + "mix.k.norm", D)
                v = self.heads(self.times(h, p + "mix.v", K), D)
                if values is None:
                    values = v
                else:
                    share = self.w(p + "mix.vmix")
                    v = (1.0 - share) * v + share * values
                o = attend(q, k, v, m["scale"], self.spans, cap=m["softcap"])
                o = o * torch.sigmoid(self.times(h, p + "mix.g", m["heads"]))[..., None]
                y = self.times(o.reshape(x.shape[0], Q), p + "mix.o", hidden)
            x = x + norm(p + "norm1b", y)
            h = norm(p + "norm2", x)
            if mlp["kind"] == "dense":
                up = torch.relu(self.times(h, p + "mlp.up", self.ff, p + "mlp.up.b")).pow(2)
                y = self.times(up, p + "mlp.down", hidden, p + "mlp.down.b")
            else:
                r = mlp["router"]
                best = self.times(h, p + "mlp.router", r["experts"], p + "mlp.router.b").topk(r["top"], -1)
                y = self.experts(p + "mlp.", mlp, h, best.indices, torch.softmax(best.values, -1))
                share = torch.sigmoid(self.times(h, p + "mlp.shared.sg", 1))
                y = y + share * self.gated(h, p + "mlp.shared.", mlp["shared"]["ff"], silu)
            x = x + norm(p + "norm2b", y)
        return self.logits(norm("final.norm", x), "head")


def exact(case, seed):
    with torch.no_grad():
        return getattr(Exact(case, seed), case["design"])()
