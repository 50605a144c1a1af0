"""What is measured when this engine's speed is: the work that programs have it do, case by case.

A case is one of two kinds. ``steps``: calls of ``Engine.step`` with tokens that are known beforehand (the scheduler's own
steps, with given tokens in the place of chosen ones, so that logits can be compared): single tokens of requests that hold
a context, prompts, prompts and what follows them, or portions of prompts beside single tokens. ``generate``: a call of
``generate``, scheduler, selection and all. Weights are drawn at random at the widths of the models that ``bench.py``
names; depth is cut where the full one would only repeat the same layer for longer.

``exact`` is a second implementation in 64 bits, whole sequences, no cache, from this file alone.
"""
from __future__ import annotations

import math
import random
import zlib
from types import SimpleNamespace

import numpy as np
import torch

QWEN2 = {
    "7b": dict(vocab=152064, width=3584, layers=28, heads=28, kv_heads=4, dim=128, ff=18944, tied=False),
    "0.5b": dict(vocab=151936, width=896, layers=24, heads=14, kv_heads=2, dim=64, ff=4864, tied=True),
}
DESIGNS = ("siditar", "zabozen", "zuluvik")
DESIGN_SIZES = {
    "1k": dict(vocab=32768, width=1024, heads=8, kv_heads=2, dim=128, ff=4096),
    "2k": dict(vocab=32768, width=2048, heads=16, kv_heads=4, dim=128, ff=8192),
}
LATENT = dict(dim=96, rot=64, rank=192, scale=160 ** -0.5)      # of the designs' latent attention
EPS = 1e-6
ROT_BASE = 1e6
RAMP = dict(factor=16.0, original=8192.0, fast=24.0, slow=1.5)  # Zuluvik's stretched rotation
EXPERTS = dict(experts=16, identity=4, top=4, limit=7.0)
EXACT_FLOPS = 2.5e14        # what 64 bits finish in well under 20 seconds
DEVICE = "cuda:0"


# ---- the cases --------------------------------------------------------------------------------------------------
def listed():
    qwen = dict(kind="steps", requests=1, context=0, shortest=0, new=0, dtype="bfloat16", portion=0)
    return [
        # A chat's next tokens, one user, the smallest model: the shortest step there is, launches and host included.
        dict(qwen, name="0.5b decode 1x60", model="0.5b", layers=24, context=60, shortest=60, new=8),
        # The headline: eight requests deep in a conversation, the whole model.
        dict(qwen, name="7b decode 8x4096", model="7b", layers=28, requests=8, context=4096, shortest=4096, new=8),
        # A busy server: 64 requests of ragged lengths, weights and caches both long to read.
        dict(qwen, name="7b decode 64x<3000", model="7b", layers=8, requests=64, context=2999, shortest=150, new=8),
        # A prompt on an idle server, the whole model.
        dict(qwen, name="7b prompt 2048", model="7b", layers=28, context=2048),
        # A document, odd in length; attention is a large part.
        dict(qwen, name="7b prompt 16301", model="7b", layers=8, context=16301),
        # Continuous batching step by step: portions of new prompts beside single tokens of the others.
        dict(qwen, name="0.5b mixed 10x<1500", model="0.5b", layers=24, requests=10, context=1500, shortest=70, new=12, portion=512),
        # The Python entry point: prompts through scheduler, steps and selection (greedy and drawn) to their tokens.
        dict(qwen, name="0.5b generate 32x<1000", kind="generate", model="0.5b", layers=24, requests=32, context=1000, shortest=100, new=48),
        # The 32-bit engine, single tokens: what an exact evaluation decodes with.
        dict(qwen, name="7b fp32 decode 8x2000", model="7b", layers=6, requests=8, context=2000, shortest=2000, new=4, dtype="float32"),
        # And its prompts: scoring a text of ordinary, odd length.
        dict(qwen, name="0.5b fp32 prompt 1003", model="0.5b", layers=24, context=1003, dtype="float32"),
        # The further designs, each as a request meets it: two prompts, then single tokens.
        dict(qwen, name="siditar 2x<2000+8", model="siditar 2k", layers=4, requests=2, context=2000, shortest=1117, new=8),
        dict(qwen, name="zabozen 2x<2000+8", model="zabozen 2k", layers=4, requests=2, context=2000, shortest=1117, new=8),
        dict(qwen, name="zuluvik 2x<2000+8", model="zuluvik 2k", layers=4, requests=2, context=2000, shortest=1117, new=8),
    ]


def draw(rng: random.Random) -> dict:
    def over(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    kind = rng.choice(("decode", "decode", "prompt", "prompt", "mixed", "design", "design", "generate"))
    case = dict(kind="steps", model=rng.choice(("0.5b", "7b")), layers=rng.randint(2, 6), requests=1, context=0, shortest=0, new=0,
                dtype=rng.choice(("bfloat16", "bfloat16", "float32")), portion=0)
    if case["model"] == "0.5b":
        case["layers"] = rng.randint(6, 24)
    if kind == "decode":
        case.update(requests=over(1, 64), new=8)
        longest = min(8192, 100_000 // case["requests"]) if case["dtype"] == "bfloat16" else min(2048, 16_000 // case["requests"])
        case["context"] = over(17, longest)
        case["shortest"] = over(16, case["context"])
    elif kind == "prompt":
        case.update(context=over(17, 16384 if case["dtype"] == "bfloat16" else 1500))
    elif kind == "mixed":
        case.update(model="0.5b", layers=rng.randint(6, 24), requests=rng.randint(3, 12), context=over(200, 1500), new=rng.randint(4, 12),
                    portion=rng.choice((128, 256, 512)), dtype="bfloat16")
        case["shortest"] = over(20, case["context"])
    elif kind == "generate":
        case.update(kind="generate", model="0.5b", layers=rng.randint(6, 24), requests=over(1, 32), context=over(60, 1000), new=rng.randint(8, 48),
                    dtype="bfloat16")
        case["shortest"] = over(16, case["context"])
    else:
        case.update(model=f"{rng.choice(DESIGNS)} {rng.choice(tuple(DESIGN_SIZES))}", layers=rng.randint(2, 4), requests=rng.randint(1, 4),
                    context=over(40, 2000), new=8, dtype="bfloat16")
        case["shortest"] = over(20, case["context"])
    return case


def contexts(case) -> list:
    """Every request's context or prompt: between the shortest and the longest, spread over the logarithm, the longest first."""
    long, short, out = case["context"], case["shortest"] or case["context"], []
    for index in range(case["requests"]):
        out.append(int(round(long * (short / long) ** ((index * 0.6180339887) % 1.0))))
    return out


def script(case):
    """``(held, steps)``: the requests' lengths before the pass, and the steps of it: per step the requests that are opened
    and a list of ``(request, first, count, wanted places)``."""
    lengths, new = contexts(case), case["new"]
    everyone = range(case["requests"])
    if case["portion"]:                         # prompts in portions, 2048 tokens a step, new requests as there is room
        steps, done, opened = [], [0] * len(lengths), 0
        while any(done[r] < lengths[r] + new for r in everyone):
            entries, room, opens = [], 2048, []
            for r in everyone:
                if r >= opened and room < case["portion"]:
                    break
                left = lengths[r] - done[r]
                if left <= 0 and done[r] >= lengths[r] + new:
                    continue
                count = min(left, case["portion"], room) if left > 0 else 1
                if count <= 0:
                    continue
                if r >= opened:
                    if len(opens) == 2:         # two arrive a step
                        break
                    opens.append(r)
                    opened = r + 1
                entries.append((r, done[r], count, (count - 1,) if done[r] + count >= lengths[r] else ()))
                done[r] += count
                room -= count
            steps.append((opens, entries))
        return None, steps
    if new and model_of(case).design is None:   # single tokens after contexts that were there before
        return lengths, [((), [(r, lengths[r] + i, 1, (0,)) for r in everyone]) for i in range(new)]
    steps = [(list(everyone), [(r, 0, lengths[r], (lengths[r] - 1,)) for r in everyone])]
    return None, steps + [((), [(r, lengths[r] + i, 1, (0,)) for r in everyone]) for i in range(new)]


# ---- weights ----------------------------------------------------------------------------------------------------
def model_of(case) -> SimpleNamespace:
    name = case["model"].split()
    sizes = dict(QWEN2[name[0]]) if len(name) == 1 else dict(DESIGN_SIZES[name[1]])
    sizes.update(layers=case["layers"], design=None if len(name) == 1 else name[0])
    if case["kind"] == "generate":
        sizes["tied"] = False
    return SimpleNamespace(**sizes)


def shapes(m) -> dict:
    """Name of every tensor in the model's file -> ``(shape, mean, standard deviation)``."""
    w, out = m.width, {}

    def matrix(name, *shape, std=0.02, mean=0.0):
        out[name] = (shape, mean, std)

    def gain(name, *shape):
        out[name] = (shape, 1.0, 0.1)

    if m.design is None:
        matrix("model.embed_tokens.weight", m.vocab, w)
        for i in range(m.layers):
            p = f"model.layers.{i}."
            gain(p + "input_layernorm.weight", w)
            gain(p + "post_attention_layernorm.weight", w)
            for role, rows in (("q", m.heads * m.dim), ("k", m.kv_heads * m.dim), ("v", m.kv_heads * m.dim)):
                matrix(p + f"self_attn.{role}_proj.weight", rows, w)
                matrix(p + f"self_attn.{role}_proj.bias", rows, std=0.2)
            matrix(p + "self_attn.o_proj.weight", w, m.heads * m.dim)
            matrix(p + "mlp.gate_proj.weight", m.ff, w)
            matrix(p + "mlp.up_proj.weight", m.ff, w)
            matrix(p + "mlp.down_proj.weight", w, m.ff)
        gain("model.norm.weight", w)
        if not m.tied:
            matrix("lm_head.weight", m.vocab, w)
        return out
    heads, kv, dim, ff = m.heads, m.kv_heads, m.dim, m.ff
    matrix("embed", m.vocab, w)
    matrix("head", m.vocab, w)
    gain("final.norm", w)

    def attention(p, biases, value_rows=kv * dim, keys=True):
        rows = {"q": heads * dim, "k": kv * dim, "v": value_rows}
        for role in ("q", "k", "v") if keys else ("q",):
            matrix(p + role, rows[role], w)
            if biases:
                matrix(p + role + ".b", rows[role], std=0.5)
        matrix(p + "o", w, heads * dim)

    def latent(p):
        matrix(p + "q", heads * (LATENT["dim"] + LATENT["rot"]), w)
        matrix(p + "dkv", LATENT["rank"] + LATENT["rot"], w)
        gain(p + "dkv.norm", LATENT["rank"])
        matrix(p + "uk", heads * LATENT["dim"], LATENT["rank"])
        matrix(p + "uv", heads * dim, LATENT["rank"])
        matrix(p + "o", w, heads * dim)

    def dense(p, inner):
        matrix(p + "gate", inner, w)
        matrix(p + "up", inner, w)
        matrix(p + "down", w, inner)

    for i in range(m.layers):
        p = f"l{i}."
        gain(p + "norm1", w)
        if m.design == "siditar":
            gain(p + "norm2", w)
            left, right, inner = p + "mix.left.", p + "mix.right.", heads // 2
            attention(left, False)
            gain(left + "q.norm", dim)
            gain(left + "k.norm", dim)
            matrix(left + "rel", 32, heads, std=0.5)
            matrix(left + "sink", heads, std=0.5)
            for role, rows in (("q", inner * dim // 2), ("k", inner * dim // 2), ("v", inner * dim), ("g", inner * dim), ("a1", 16)):
                matrix(right + role, rows, w)
            matrix(right + "o", w, inner * dim)
            gain(right + "norm", dim)
            matrix(right + "a2", inner * dim // 2, 16, std=0.2)
            matrix(right + "a2.b", inner * dim // 2, std=0.5)
            dense(p + "mlp.", ff)
            for joint in ("hc1", "hc2"):
                matrix(p + joint + ".in", 2, mean=0.5, std=0.1)
                matrix(p + joint + ".out", 2, mean=1.0, std=0.1)
                matrix(p + joint + ".mix", 2, 2, mean=0.5, std=0.1)
        elif m.design == "zabozen":
            for norm in ("norm1b", "norm2", "norm2b"):
                gain(p + norm, w)
            if i % 4 == 0:
                latent(p + "mix.")
                matrix(p + "mix.g", heads, w)
            elif i % 4 == 1:
                for role, rows in (("q", kv * dim), ("k", kv * dim), ("v", heads * dim)):
                    matrix(p + f"mix.{role}", rows, w)
                    matrix(p + f"mix.{role}.conv", rows, 4, std=0.3)
                matrix(p + "mix.g", heads * dim, w)
                matrix(p + "mix.a", heads, w)
                matrix(p + "mix.b", heads, w)
                matrix(p + "mix.dt_bias", heads, std=0.5)
                matrix(p + "mix.A_log", heads, std=0.5)
                gain(p + "mix.norm", dim)
                matrix(p + "mix.o", w, heads * dim)
            else:
                attention(p + "mix.", True, keys=i % 4 == 2)
                matrix(p + "mix.o.b", w, std=0.5)
            dense(p + "mlp.", ff)
        else:
            if i % 4 == 0:
                attention(p + "mix.", False)
                for role, rows in (("q", heads * dim), ("k", kv * dim), ("v", kv * dim)):
                    matrix(p + f"mix.{role}.conv", rows, 4, std=0.3)
                for name in ("lq1", "lk1", "lq2", "lk2"):
                    matrix(p + "mix." + name, dim // 2, std=0.1)
            elif i % 4 == 2:
                latent(p + "mix.")
            else:
                attention(p + "mix.", True)
            # Wide router scores, as training gives them: the last of the chosen has little weight, so that a tie in the
            # choice (which rounding may decide either way) moves the result little.
            matrix(p + "mlp.router", EXPERTS["experts"] + EXPERTS["identity"], w, std=0.1)
            matrix(p + "mlp.correction", EXPERTS["experts"] + EXPERTS["identity"], std=0.001)
            for expert in range(EXPERTS["experts"]):
                dense(p + f"mlp.e{expert}.", ff // 4)
            dense(p + "mlp.shared.", ff // 2)
    return out


def draw_weights(case, seed: int) -> dict:
    """The model's tensors in bfloat16, every one from a generator of its own."""
    m, out = model_of(case), {}
    generator = torch.Generator(device=DEVICE)
    for name, (shape, mean, std) in shapes(m).items():
        generator.manual_seed((seed * 0x9E3779B1 + zlib.crc32(name.encode())) & 0x7FFFFFFFFFFF)
        out[name] = torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(mean, std, generator=generator)
    if case["kind"] == "generate":
        # A model that is sure of its next token, as trained ones mostly are: rounding then does not choose another one.
        embedding = out["model.embed_tokens.weight"]
        embedding.mul_(50.0)
        out["lm_head.weight"] = (torch.roll(embedding, 7919, 0) * 0.05).contiguous()
    return out


def draw_tokens(case, seed: int) -> list:
    rng = np.random.default_rng(seed + 77)
    return [rng.integers(0, model_of(case).vocab, size=length + case["new"]).tolist() for length in contexts(case)]


# ---- the pass ---------------------------------------------------------------------------------------------------
def build_config(case):
    m = model_of(case)
    if m.design is None:
        from microllm_rocm_amd import Qwen2Config
        return Qwen2Config(vocab_size=m.vocab, hidden_size=m.width, num_hidden_layers=m.layers, num_attention_heads=m.heads,
                           num_key_value_heads=m.kv_heads, head_dim=m.dim, intermediate_size=m.ff, max_position_embeddings=32768,
                           rope_theta=ROT_BASE, rms_norm_eps=EPS, tie_word_embeddings=m.tied)
    if m.design == "siditar":
        from microllm_rocm_amd.config.siditar import (BiasAttentionConfig, DenseMlpConfig, LinearAttentionConfig, ParallelMixerConfig,
                                                      SiditarConfig, SiditarLayerConfig)
        left = BiasAttentionConfig(heads=m.heads, kv_heads=m.kv_heads, dim=m.dim, vdim=m.dim, scale=m.dim ** -0.5, bias_max=1024,
                                   temp_coef=0.5, temp_every=64, bias_rows=32)
        right = LinearAttentionConfig(heads=m.heads // 2, dim=m.dim // 2, vdim=m.dim, tau=16.0, decay_rank=16)
        layer = SiditarLayerConfig("parallel", ParallelMixerConfig(left, right, 1.0, 1.0), DenseMlpConfig(m.ff, 7.0))
        return SiditarConfig(vocab=m.vocab, width=m.width, norm_eps=EPS, layers=(layer,) * m.layers, streams=2)
    if m.design == "zabozen":
        from microllm_rocm_amd.config.zabozen import (DeltaConfig, DenseMlpConfig, LatentAttentionConfig, WindowAttentionConfig,
                                                      ZabozenConfig, ZabozenLayerConfig)
        latent = LatentAttentionConfig(heads=m.heads, dim=LATENT["dim"], rot_dim=LATENT["rot"], vdim=m.dim, kv_rank=LATENT["rank"],
                                       scale=LATENT["scale"], rot_base=ROT_BASE, rot_dims=LATENT["rot"])
        delta = DeltaConfig(heads=m.heads, kv_heads=m.kv_heads, dim=m.dim, vdim=m.dim, conv=4)
        layers = []
        for i in range(m.layers):
            window = WindowAttentionConfig(heads=m.heads, kv_heads=m.kv_heads, dim=m.dim, vdim=m.dim, scale=m.dim ** -0.5, window=1024,
                                           kv_from=i - 1 if i % 4 == 3 else None)
            kind, mixer = (("latent_attention", latent), ("delta", delta), ("attention", window), ("attention", window))[i % 4]
            layers.append(ZabozenLayerConfig(kind, mixer, DenseMlpConfig(m.ff)))
        return ZabozenConfig(vocab=m.vocab, width=m.width, norm_eps=EPS, residual_mult=0.5, layers=tuple(layers), logit_softcap=30.0)
    from microllm_rocm_amd.config.zuluvik import (DifferentialAttentionConfig, ExpertConfig, LatentAttentionConfig, MoeMlpConfig,
                                                  RampScalingConfig, RotaryAttentionConfig, RotationConfig, ZuluvikConfig, ZuluvikLayerConfig)
    scaling = RampScalingConfig(**RAMP)
    differential = DifferentialAttentionConfig(heads=m.heads, kv_heads=m.kv_heads, dim=m.dim // 2, vdim=m.dim, conv=4, diff=0.7,
                                               scale=(m.dim // 2) ** -0.5)
    rotary = RotaryAttentionConfig(heads=m.heads, kv_heads=m.kv_heads, dim=m.dim, vdim=m.dim, scale=m.dim ** -0.5,
                                   rot=RotationConfig(ROT_BASE, m.dim // 2, scaling))
    latent = LatentAttentionConfig(heads=m.heads, dim=LATENT["dim"], rot_dim=LATENT["rot"], vdim=m.dim, kv_rank=LATENT["rank"],
                                   scale=LATENT["scale"], rot=RotationConfig(ROT_BASE, LATENT["rot"], scaling))
    moe = MoeMlpConfig(experts=EXPERTS["experts"], top=EXPERTS["top"], expert=ExpertConfig(m.ff // 4, EXPERTS["limit"]),
                       identity=EXPERTS["identity"], scale=1.0, shared=ExpertConfig(m.ff // 2, EXPERTS["limit"]))
    kinds = (("attention", differential), ("attention_2", rotary), ("latent_attention", latent), ("attention_2", rotary))
    return ZuluvikConfig(vocab=m.vocab, width=m.width, norm_eps=EPS, layers=tuple(ZuluvikLayerConfig(*kinds[i % 4], moe) for i in range(m.layers)),
                         embedding_scale=m.width ** 0.5)


def prepare(case, seed):
    from microllm_rocm_amd import Engine, SamplingParams, StepEntry
    from microllm_rocm_amd.config.registry import architecture_named
    config = build_config(case)
    tokens = draw_tokens(case, seed)
    engine = Engine(architecture_named(config.architecture).build_spec(config), draw_weights(case, seed), dtype=case["dtype"], device=DEVICE,
                    max_tokens=sum(-(-len(t) // 16) * 16 + 16 for t in tokens), max_requests=max(4, case["requests"]), consume_tensors=True)
    state = SimpleNamespace(engine=engine)
    if case["kind"] == "generate":
        state.prompts = [t[:length] for t, length in zip(tokens, contexts(case))]
        # every other request draws its tokens, the others take the most likely one
        state.params = [SamplingParams(max_new_tokens=case["new"], temperature=0.8 if index % 2 else 0.0, top_k=40 if index % 4 == 1 else 0,
                                       seed=index) for index in range(case["requests"])]
        return state
    held, steps = script(case)
    state.held = None
    if held is not None:
        waiting = []
        for request, length in enumerate(held):
            engine.open(request)
            waiting.append(StepEntry(request, tokens[request][:length]))
            if sum(len(entry.tokens) for entry in waiting) > 8192 or request == len(held) - 1:
                engine.step(waiting)
                waiting = []
        state.held = [(engine.cache.get(request), length) for request, length in enumerate(held)]
    state.steps = [(list(opens), [StepEntry(r, tokens[r][first:first + count], want) for r, first, count, want in entries])
                   for opens, entries in steps]
    state.opened = [request for opens, _ in state.steps for request in opens]
    return state


def run(state):
    """``steps``: the logits of every step that wants any; ``generate``: every request's prompt and new tokens."""
    engine = state.engine
    if not hasattr(state, "steps"):
        from microllm_rocm_amd import generate
        return [np.asarray(tokens) for tokens in generate(engine, state.prompts, state.params)]
    out = []
    for opens, entries in state.steps:
        for request in opens:
            engine.open(request)
        logits = engine.step(entries)
        if logits is not None:
            out.append(logits)
    for request in state.opened:
        engine.close(request)
    if state.held is not None:      # what was scored is taken back: lengths, not contents, say what is valid
        for request, length in state.held:
            request.num_tokens = length
            engine.cache.cancel_reservation(request)
    return out


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def work(case):
    m = model_of(case)
    size = 4 if case["dtype"] == "float32" else 2
    sizes = {name: math.prod(shape) for name, (shape, _, _) in shapes(m).items()}
    embedding = "model.embed_tokens.weight" if m.design is None else "embed"
    head = embedding if m.design is None and m.tied else ("lm_head.weight" if m.design is None else "head")
    experts = sum(count for name, count in sizes.items() if ".mlp.e" in name)
    layers = sum(count for name, count in sizes.items() if name not in (embedding, head)) - experts
    attending = m.layers if m.design != "zabozen" else sum(1 for i in range(m.layers) if i % 4 != 1)
    per_key = m.heads * m.dim * 4                           # flops: scores and values
    per_position = 2 * m.kv_heads * m.dim * size            # bytes of a layer's keys and values
    if case["kind"] == "generate":
        lengths = contexts(case)
        steps = [([], [(r, 0, length, (length - 1,)) for r, length in enumerate(lengths)])]
        steps += [([], [(r, length + i, 1, (0,)) for r, length in enumerate(lengths)]) for i in range(case["new"] - 1)]
    else:
        _, steps = script(case)
    total_bytes = total_flops = 0.0
    for _, entries in steps:
        rows = sum(count for _, _, count, _ in entries)
        wanted = sum(len(want) for _, _, _, want in entries)
        reached = min(1.0, rows * EXPERTS["top"] / EXPERTS["experts"])
        active = EXPERTS["top"] / (EXPERTS["experts"] + EXPERTS["identity"])
        total_bytes += (layers + experts * reached + (sizes[head] if wanted else 0) + rows * m.width) * size + wanted * m.vocab * 4
        total_flops += 2.0 * rows * (layers + experts * active) + 2.0 * wanted * sizes[head]
        for _, first, count, _ in entries:
            keys = first + count
            total_bytes += attending * (keys + (count if first else 0)) * per_position
            total_flops += attending * per_key * (count * first + count * (count + 1) / 2)
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """Four times the distance from ``exact`` that this engine's logits have: 1.1e-6 to 4.3e-6 in float32; in bfloat16 4e-3 to
    1.8e-2, the deepest model the furthest (where four times is more than the format should need: 0.03). Tokens are chosen
    by a wide margin; one that a tie decides changes the rest of its request."""
    if case["kind"] == "generate":
        return {"differ": 0.002}
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "generate":
        return None
    lengths, new = contexts(case), case["new"]
    flops = work(case)["flops"]
    if script(case)[0] is not None:     # the contexts are computed here too
        flops += work(dict(case, new=0))["flops"]
    if flops > EXACT_FLOPS:
        return None
    weights = draw_weights(case, seed)
    sequences = [t[:length + new] for t, length in zip(draw_tokens(case, seed), lengths)]
    wanted = [[] for _ in sequences]        # places whose logits a step wants, in the order of the steps
    where = []
    for _, entries in script(case)[1]:
        rows = []
        for r, first, _, want in entries:
            for place in want:
                rows.append((r, len(wanted[r])))
                wanted[r].append(first + place)
        if rows:
            where.append(rows)
    with torch.no_grad():
        logits = _Exact(model_of(case), weights).logits(sequences, wanted)
    return [torch.stack([logits[r][row] for r, row in rows]) for rows in where]


def _rms(a, weight=None):
    a = a / torch.sqrt((a * a).mean(-1, keepdim=True) + EPS)
    return a if weight is None else a * weight


def _layer_norm(a, weight):
    a = a - a.mean(-1, keepdim=True)
    return a / torch.sqrt((a * a).mean(-1, keepdim=True) + EPS) * weight


def _silu(a):
    return a * torch.sigmoid(a)


def _turn(a, rates, neighbours=False, factor=1.0):
    """``a [T, heads, n]``, every pair of the ``n`` dims turned by its position times its rate."""
    angle = torch.arange(a.shape[0], dtype=torch.float64, device=a.device)[:, None] * rates[None, :]
    cos, sin = torch.cos(angle)[:, None] * factor, torch.sin(angle)[:, None] * factor
    if neighbours:
        u, v = a[..., 0::2], a[..., 1::2]
        return torch.stack([u * cos - v * sin, v * cos + u * sin], dim=-1).reshape(a.shape)
    u, v = a.chunk(2, dim=-1)
    return torch.cat([u * cos - v * sin, v * cos + u * sin], dim=-1)


def _rates(n, device, ramp=None):
    pairs = torch.arange(n // 2, dtype=torch.float64, device=device)
    rates = ROT_BASE ** (-2.0 * pairs / n)
    if ramp is None:
        return rates, 1.0

    def pair(times):
        return n * math.log(ramp["original"] / (2.0 * math.pi * times)) / (2.0 * math.log(ROT_BASE))

    low, high = max(math.floor(pair(ramp["fast"])), 0), min(math.ceil(pair(ramp["slow"])), n - 1)
    blend = ((pairs - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
    return rates / ramp["factor"] * blend + rates * (1.0 - blend), 0.1 * math.log(ramp["factor"]) + 1.0


def _attend(q, k, v, scale, window=None, bias=None, sink=None):
    """``q [T, H, d]``, ``k [T, G, d]``, ``v [T, G, dv]``, query ``i`` over the keys ``j <= i``; ``bias(distance, heads)`` is
    added to the scores, ``sink [H]`` is one more score that has no value."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    block, group = 1024, H // G
    places = torch.arange(T, device=q.device)
    for start in range(0, T, block):
        stop = min(T, start + block)
        first = 0 if window is None else max(0, start - window + 1)
        distance = places[start:stop, None] - places[None, first:stop]
        hidden = distance < 0 if window is None else (distance < 0) | (distance >= window)
        for g in range(G):
            heads = slice(g * group, (g + 1) * group)
            scores = (q[start:stop, heads].transpose(0, 1) @ k[first:stop, g].T) * scale
            if bias is not None:
                scores += bias(distance, heads)
            scores.masked_fill_(hidden, float("-inf"))
            top = scores.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[heads][:, None, None])
            scores = torch.exp(scores.sub_(top))
            total = scores.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[heads][:, None, None] - top)
            out[start:stop, heads] = ((scores @ v[first:stop, g]) / total).transpose(0, 1)
    return out


def _convolve(a, taps):
    n = taps.shape[1]
    padded = torch.cat([a.new_zeros(n - 1, a.shape[1]), a])
    return sum(taps[:, j] * padded[j:j + a.shape[0]] for j in range(n))


class _Exact:
    def __init__(self, m, weights):
        self.m, self.weights = m, weights

    def w(self, name):
        return self.weights[name].to(torch.float64)

    def product(self, a, name, bias=False):
        out = a @ self.w(name).T
        return out + self.w(name + ".b") if bias else out

    def logits(self, sequences, wanted):
        m = self.m
        ids = [torch.tensor(s, device=DEVICE) for s in sequences]
        bounds = np.cumsum([0] + [len(s) for s in sequences]).tolist()
        self.pieces = list(zip(bounds[:-1], bounds[1:]))
        rows = torch.cat([torch.tensor(places, device=DEVICE, dtype=torch.int64) + start for places, (start, _) in zip(wanted, self.pieces)])
        embedding = self.weights["model.embed_tokens.weight" if m.design is None else "embed"]
        x = embedding[torch.cat(ids)].to(torch.float64)
        x = getattr(self, m.design or "qwen2")(x)
        if m.design is None:
            out = _rms(x[rows], self.w("model.norm.weight")) @ self.w("model.embed_tokens.weight" if m.tied else "lm_head.weight").T
        elif m.design == "siditar":
            out = _layer_norm(x[rows], self.w("final.norm")) @ self.w("head").T
        else:
            out = _rms(x[rows], self.w("final.norm")) @ self.w("head").T
            if m.design == "zabozen":
                out = 30.0 * torch.tanh(out / 30.0)
        return out.split([len(places) for places in wanted])

    def each(self, function, *tensors):
        """``function`` on every sequence's rows of the given tensors; the results under one another again."""
        return torch.cat([function(*(t[a:b] for t in tensors)) for a, b in self.pieces])

    def qwen2(self, x):
        m = self.m
        rates, _ = _rates(m.dim, x.device)

        def attend(q, k, v):
            T = q.shape[0]
            return _attend(_turn(q.view(T, m.heads, m.dim), rates), _turn(k.view(T, m.kv_heads, m.dim), rates),
                           v.view(T, m.kv_heads, m.dim), m.dim ** -0.5).reshape(T, -1)

        for i in range(m.layers):
            p = f"model.layers.{i}."
            a = _rms(x, self.w(p + "input_layernorm.weight"))
            q, k, v = (a @ self.w(p + f"self_attn.{r}_proj.weight").T + self.w(p + f"self_attn.{r}_proj.bias") for r in "qkv")
            x = x + self.each(attend, q, k, v) @ self.w(p + "self_attn.o_proj.weight").T
            a = _rms(x, self.w(p + "post_attention_layernorm.weight"))
            hidden = _silu(a @ self.w(p + "mlp.gate_proj.weight").T).mul_(a @ self.w(p + "mlp.up_proj.weight").T)
            x = x + hidden @ self.w(p + "mlp.down_proj.weight").T
        return x

    def siditar(self, x):
        m = self.m
        columns = torch.arange(m.width, device=x.device)
        rates = 10000.0 ** (-2.0 * (columns // 2).to(torch.float64) / m.width)

        def waves(rows):
            angle = torch.arange(rows.shape[0], device=x.device, dtype=torch.float64)[:, None] * rates
            return torch.where(columns % 2 == 1, torch.cos(angle), torch.sin(angle))

        x = x + self.each(waves, x)
        streams = [x, x]
        for i in range(m.layers):
            p = f"l{i}."
            for number, sublayer in (("1", self.siditar_mixer), ("2", self.siditar_feed_forward)):
                joint = p + "hc" + number
                take, give, mix = self.w(joint + ".in"), self.w(joint + ".out"), self.w(joint + ".mix")
                y = sublayer(_layer_norm(take[0] * streams[0] + take[1] * streams[1], self.w(p + "norm" + number)), p)
                streams = [mix[0, t] * streams[0] + mix[1, t] * streams[1] + give[t] * y for t in (0, 1)]
        return streams[0] + streams[1]

    def siditar_feed_forward(self, a, p):
        gate = torch.clamp(self.product(a, p + "mlp.gate"), max=7.0)
        up = torch.clamp(self.product(a, p + "mlp.up"), -7.0, 7.0)
        return self.product(gate * torch.sigmoid(1.702 * gate) * (up + 1.0), p + "mlp.down")

    def siditar_mixer(self, a, p):
        m = self.m
        left, right, inner, small = p + "mix.left.", p + "mix.right.", m.heads // 2, m.dim // 2
        table, sink = self.w(left + "rel"), self.w(left + "sink")
        buckets = []
        for distance in range(1025):
            buckets.append(distance if distance < 16 else min(31, 16 + int(math.floor(math.log(distance / 16) / math.log(1024 / 16) * 16))))
        unrolled = table[torch.tensor(buckets, device=a.device)]            # [distance, heads]

        def attend(q, k, v):
            T = q.shape[0]
            factor = 1.0 + 0.5 * torch.log((torch.arange(T, device=q.device) + 1) // 64 + torch.ones((), dtype=torch.float64, device=q.device))
            q = _rms(q.view(T, m.heads, m.dim), self.w(left + "q.norm")) * factor[:, None, None]
            k = _rms(k.view(T, m.kv_heads, m.dim), self.w(left + "k.norm"))
            return _attend(q, k, v.view(T, m.kv_heads, m.dim), m.dim ** -0.5, sink=sink,
                           bias=lambda distance, heads: unrolled[distance.clamp(0, 1024)][..., heads].permute(2, 0, 1)).reshape(T, -1)

        def walk(q, k, v, decay):
            T = q.shape[0]
            q, k, decay = (t.reshape(T, inner, small) for t in (q, k, decay))
            v = v.reshape(T, inner, m.dim)
            state, out = q.new_zeros(inner, small, m.dim), torch.empty(T, inner, m.dim, dtype=q.dtype, device=q.device)
            for t in range(T):
                state = decay[t, :, :, None] * state + k[t, :, :, None] * v[t, :, None, :]
                out[t] = (state * q[t, :, :, None]).sum(1)
            return out.reshape(T, -1)

        out = self.product(self.each(attend, *(self.product(a, left + role) for role in "qkv")), left + "o")
        z = self.product(self.product(a, right + "a1"), right + "a2") + self.w(right + "a2.b")
        decay = torch.sigmoid(z) ** (1.0 / 16.0)
        o = self.each(walk, self.product(a, right + "q") * small ** -0.5, self.product(a, right + "k"), self.product(a, right + "v"), decay)
        o = _rms(o.view(-1, inner, m.dim), self.w(right + "norm")).reshape(o.shape)
        return out + self.product(o * _silu(self.product(a, right + "g")), right + "o")

    def latent(self, a, p, neighbours, ramp):
        m, c = self.m, LATENT
        rates, factor = _rates(c["rot"], a.device, ramp)

        def attend(q, down):
            T = q.shape[0]
            q = q.view(T, m.heads, c["dim"] + c["rot"])
            q = torch.cat([q[..., :c["dim"]], _turn(q[..., c["dim"]:], rates, neighbours, factor)], dim=-1)
            latent = _rms(down[:, :c["rank"]], self.w(p + "dkv.norm"))
            turned = _turn(down[:, None, c["rank"]:], rates, neighbours, factor)
            keys = torch.cat([self.product(latent, p + "uk").view(T, m.heads, c["dim"]), turned.expand(T, m.heads, c["rot"])], dim=-1)
            return _attend(q, keys, self.product(latent, p + "uv").view(T, m.heads, m.dim), c["scale"]).reshape(T, -1)

        return self.each(attend, self.product(a, p + "q"), self.product(a, p + "dkv"))

    def zabozen(self, x):
        m = self.m
        kept = None
        slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / m.heads) for h in range(m.heads)], dtype=torch.float64, device=x.device)

        def attend(q, k, v):
            T = q.shape[0]
            return _attend(_rms(q.view(T, m.heads, m.dim)), _rms(k.view(T, m.kv_heads, m.dim)), v.view(T, m.kv_heads, m.dim), m.dim ** -0.5,
                           window=1024, bias=lambda distance, heads: -slopes[heads][:, None, None] * distance).reshape(T, -1)

        for i in range(m.layers):
            p = f"l{i}."
            a = _rms(x, self.w(p + "norm1"))
            if i % 4 == 0:
                o = self.latent(a, p + "mix.", False, None)
                gate = torch.sigmoid(self.product(a, p + "mix.g"))
                y = self.product((o.view(-1, m.heads, m.dim) * gate[:, :, None]).reshape(o.shape), p + "mix.o")
            elif i % 4 == 1:
                y = self.delta(a, p + "mix.")
            else:
                if i % 4 == 2:
                    kept = (self.product(a, p + "mix.k", True), self.product(a, p + "mix.v", True))
                y = self.product(self.each(attend, self.product(a, p + "mix.q", True), *kept), p + "mix.o", True)
            x = x + 0.5 * _rms(y, self.w(p + "norm1b"))
            a = _rms(x, self.w(p + "norm2"))
            hidden = _silu(self.product(a, p + "mlp.gate")) * self.product(a, p + "mlp.up")
            x = x + 0.5 * _rms(self.product(hidden, p + "mlp.down"), self.w(p + "norm2b"))
        return x

    def delta(self, a, p):
        m = self.m
        group = m.heads // m.kv_heads

        def walk(q, k, v, beta, decay):
            T = q.shape[0]
            q, k, v = (_silu(_convolve(t, self.w(p + f"{role}.conv"))) for role, t in (("q", q), ("k", k), ("v", v)))
            q, k = (t.view(T, m.kv_heads, m.dim) for t in (q, k))
            q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            q, k = (q * m.dim ** -0.5).repeat_interleave(group, 1), k.repeat_interleave(group, 1)
            v = v.view(T, m.heads, m.dim)
            state, out = q.new_zeros(m.heads, m.dim, m.dim), torch.empty(T, m.heads, m.dim, dtype=q.dtype, device=q.device)
            for t in range(T):
                state = decay[t, :, None, None] * state
                u = beta[t, :, None] * (v[t] - (state * k[t, :, :, None]).sum(1))
                state = state + k[t, :, :, None] * u[:, None, :]
                out[t] = (state * q[t, :, :, None]).sum(1)
            return out

        beta = torch.sigmoid(self.product(a, p + "b"))
        step = torch.nn.functional.softplus(self.product(a, p + "a") + self.w(p + "dt_bias"))
        decay = torch.exp(-torch.exp(self.w(p + "A_log")) * step)
        o = _rms(self.each(walk, *(self.product(a, p + role) for role in "qkv"), beta, decay), self.w(p + "norm"))
        gate = _silu(self.product(a, p + "g"))
        return self.product(o.reshape(gate.shape) * gate, p + "o")

    def zuluvik(self, x):
        m = self.m
        x = x * m.width ** 0.5
        rates, factor = _rates(m.dim // 2, x.device, RAMP)
        for i in range(m.layers):
            p = f"l{i}."
            a = _rms(x, self.w(p + "norm1"))
            if i % 4 == 0:
                lam = (torch.exp((self.w(p + "mix.lq1") * self.w(p + "mix.lk1")).sum()) -
                       torch.exp((self.w(p + "mix.lq2") * self.w(p + "mix.lk2")).sum()) + 0.7)

                def differ(q, k, v, p=p, lam=lam):
                    T, half = q.shape[0], m.dim // 2
                    q, k, v = (_convolve(t, self.w(p + f"mix.{role}.conv")) for role, t in (("q", q), ("k", k), ("v", v)))
                    q, k, v = q.view(T, m.heads, 2, half), k.view(T, m.kv_heads, 2, half), v.view(T, m.kv_heads, m.dim)
                    one, two = (_attend(q[:, :, n], k[:, :, n], v, half ** -0.5) for n in (0, 1))
                    return (_rms(one - lam * two) * (1.0 - 0.7)).reshape(T, -1)

                o = self.each(differ, *(self.product(a, p + f"mix.{role}") for role in "qkv"))
            elif i % 4 == 2:
                o = self.latent(a, p + "mix.", True, RAMP)
            else:
                def rotary(q, k, v):
                    T, turned = q.shape[0], m.dim // 2
                    q, k, v = q.view(T, m.heads, m.dim), k.view(T, m.kv_heads, m.dim), v.view(T, m.kv_heads, m.dim)
                    q, k = (_rms(torch.cat([_turn(t[..., :turned], rates, True, factor), t[..., turned:]], dim=-1)) for t in (q, k))
                    return _attend(q, k, v, m.dim ** -0.5).reshape(T, -1)

                o = self.each(rotary, *(self.product(a, p + f"mix.{role}", True) for role in "qkv"))
            x = x + self.product(o, p + "mix.o") + self.experts(a, p + "mlp.")
        return x

    def expert(self, a, p):
        gate = torch.clamp(self.product(a, p + "gate"), max=EXPERTS["limit"])
        up = torch.clamp(self.product(a, p + "up"), -EXPERTS["limit"], EXPERTS["limit"])
        return self.product(gate * torch.sigmoid(1.702 * gate) * (up + 1.0), p + "down")

    def experts(self, a, p):
        scores = torch.softmax(self.product(a, p + "router"), dim=-1)
        chosen = torch.topk(scores + self.w(p + "correction"), EXPERTS["top"], dim=-1).indices
        weight = torch.zeros_like(scores).scatter_(1, chosen, scores.gather(1, chosen))
        weight = weight / (weight.sum(-1, keepdim=True) + 1e-20)
        out = a * weight[:, EXPERTS["experts"]:].sum(-1, keepdim=True) + self.expert(a, p + "shared.")
        for index in range(EXPERTS["experts"]):
            took = weight[:, index].nonzero()[:, 0]
            out[took] += weight[took, index, None] * self.expert(a[took], p + f"e{index}.")
        return out
