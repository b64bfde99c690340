"""The work that users of the engine have it do, as a list of cases that can be timed and checked.

Nearly every case is ONE step of a model through the engine's step function (``ModelRunner.step``, what ``Engine.step`` and
the trace replay both call): some requests that decode one token each behind contexts of their own, portions of
prompts beside them, or only one of the two.  Logits come back for every row that an engine would sample from.
The remaining case is the batched sampler behind such a step.

Models: the Qwen2.5 shapes that ``bench.py`` is quoted on and four of its other designs, which among them hold every kind of
mixer (attention over whole contexts, windows and latents, the delta rules, gated recurrences, a state space) and
feed-forward (dense, experts), at the layer sizes that ``bench.py`` gives them.  The depth is cut so that a model is quickly
made; widths, heads, experts and vocabularies are not.

A case's keys: ``model``, ``layers`` (Qwen2 only: the other designs have their own list), ``dtype``; ``decodes`` requests behind
contexts from ``low`` to ``high`` tokens (spread evenly over the logarithm); ``portions`` prompts of ``shortest`` to
``longest`` tokens, each behind ``behind`` tokens of the same prompt that an earlier step has read.  For the sampler:
``rows``, ``vocab``, ``temperature``, ``top_p``, ``top_k``, ``greedy`` (one row in so many takes the best token; 0: none).
"""
from __future__ import annotations

import math
import random
import zlib

import torch

from velox_amd import SamplingParams
from velox_amd.cache.manager import CacheManager
from velox_amd.config.registry import config_from_dict, get_architecture
from velox_amd.engine import ModelRunner, StepEntry
from velox_amd.kernels import load_ops
from velox_amd.parts.model import DecoderModel
from velox_amd.sampling.sampler import Sampler
from velox_amd.weights.loader import bind, expected_names

DEVICE = "cuda:0"
PAGE = 16
READ_CHUNK = 4096  # tokens a step brings while prepare() reads contexts
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}

# ----------------------------------------------------------------------------------------------------------------------
# models
# ----------------------------------------------------------------------------------------------------------------------
SIZES = {
    "qwen2-1.5b": dict(design="qwen2", width=1536, heads=12, kv_heads=2, dim=128, ff=8960, vocab=151936, tied=True),
    "qwen2-7b": dict(design="qwen2", width=3584, heads=28, kv_heads=4, dim=128, ff=18944, vocab=152064, tied=False),
    "tiverax-4k": dict(design="tiverax", width=4096, heads=32, dim=96, rot_dim=32, vdim=128, kv_rank=224, ff=11008, experts=32, top=4, expert_ff=1408, shared_ff=2816, vocab=32000),
    "gosulorn-2k": dict(design="gosulorn", width=2048, streams=4, ff=5632, heads=16, kv_heads=4, dim=128, window=1024, right_heads=8, gla_heads=8, gla_vdim=256, delta_heads=16,
                        delta_kv_heads=8, rank=64, vocab=32000),
    "gosulorn-4k": dict(design="gosulorn", width=4096, streams=4, ff=11008, heads=32, kv_heads=8, dim=128, window=2048, right_heads=16, gla_heads=16, gla_vdim=256, delta_heads=32,
                        delta_kv_heads=16, rank=128, vocab=32000),
    "kedanex-2k": dict(design="kedanex", width=2048, delta_heads=32, delta_dim=64, rank=64, gru_width=3072, heads=16, kv_heads=4, dim=128, window=1024, ff=8448, experts=16, top=2,
                       expert_ff=1408, vocab=32000),
    "kedanex-4k": dict(design="kedanex", width=4096, delta_heads=64, delta_dim=64, rank=128, gru_width=6144, heads=32, kv_heads=8, dim=128, window=2048, ff=16512, experts=32, top=4,
                       expert_ff=1408, vocab=32000),
    "kukulorn-2k": dict(design="kukulorn", width=2048, heads=16, kv_heads=4, dim=128, window=1024, keep_first=64, buckets=32, far=1024, space_heads=32, state=128, space_vdim=64,
                        groups=1, ff=5632, vocab=32000),
    "kukulorn-4k": dict(design="kukulorn", width=4096, heads=32, kv_heads=8, dim=128, window=2048, keep_first=64, buckets=32, far=2048, space_heads=64, state=128, space_vdim=64,
                        groups=8, ff=11008, vocab=32000),
}


def model_config(model: str, layers: int) -> dict:
    """The dictionary that the model's ``config.json`` would hold."""
    s = SIZES[model]
    if s["design"] == "qwen2":
        return {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "num_hidden_layers": layers, "hidden_size": s["width"], "num_attention_heads": s["heads"],
                "num_key_value_heads": s["kv_heads"], "intermediate_size": s["ff"], "vocab_size": s["vocab"], "rope_theta": 1000000.0, "rms_norm_eps": 1e-6,
                "tie_word_embeddings": s["tied"], "use_sliding_window": False, "max_position_embeddings": 32768}
    out = {"vocab": s["vocab"], "width": s["width"], "norm": {"eps": 1e-5}}
    dense = {"kind": "dense", "ff": s["ff"]}
    if s["design"] == "tiverax":
        mixer = {"heads": s["heads"], "dim": s["dim"], "rot_dim": s["rot_dim"], "vdim": s["vdim"], "kv_rank": s["kv_rank"], "scale": (s["dim"] + s["rot_dim"]) ** -0.5,
                 "rot": {"dims": s["rot_dim"], "base": 1e6, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
        routed = {"kind": "moe", "router": {"experts": s["experts"], "top": s["top"]}, "expert": {"ff": s["expert_ff"]}, "shared": {"ff": s["shared_ff"]}}
        # layers 2, 3 read the caches of 0, 1 and layers 6, 7 those of 4, 5
        rows = [{"type": "latent_attention", "mixer": dict(mixer, kv_from=i - 2) if i % 4 >= 2 else dict(mixer), "mlp": routed if i % 2 else dense} for i in range(8)]
        return dict(out, architecture="Tiverax", embedding={"scale": s["width"] ** 0.5}, layers=rows)
    if s["design"] == "gosulorn":
        d = s["dim"]
        left = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5, "conv": 4, "mask": {"size": s["window"]},
                "rot": {"dims": d // 2, "base": 1e6, "scaling": {"factor": 4.0}}}
        right = {"heads": s["right_heads"], "kv_heads": s["right_heads"], "dim": d, "vdim": d, "conv": 4, "a1_rank": s["rank"], "g1_rank": s["rank"]}
        kinds = {"parallel": {"left": left, "right": right, "left_scale": 0.8, "right_scale": 1.1},
                 "gla": {"heads": s["gla_heads"], "dim": d, "vdim": s["gla_vdim"], "tau": 16.0, "a1_rank": s["rank"]},
                 "delta": {"heads": s["delta_heads"], "kv_heads": s["delta_kv_heads"], "dim": d, "vdim": d, "conv": 4}}
        rows = [{"type": kind, "mixer": kinds[kind], "mlp": dense} for kind in ("parallel", "gla", "parallel", "delta") * 2]
        return dict(out, architecture="Gosulorn", streams=s["streams"], layers=rows)
    if s["design"] == "kedanex":
        delta = {"heads": s["delta_heads"], "dim": s["delta_dim"], "w1_rank": s["rank"]}
        attention = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"], "scale": s["dim"] ** -0.5, "mask": {"size": s["window"]},
                     "rot": {"dims": s["dim"], "base": 1e6}}
        routed = {"kind": "moe", "router": {"experts": s["experts"], "top": s["top"]}, "expert": {"ff": s["expert_ff"]}}
        order = (("general_delta", delta, dense), ("mingru", {"width": s["gru_width"]}, routed), ("attention", attention, routed), ("general_delta", delta, routed))
        rows = [{"type": kind, "mixer": mixer, "mlp": mlp} for kind, mixer, mlp in order * 2]
        rows[7]["weights_of"] = 3
        return dict(out, architecture="Kedanex", norm={"eps": 1e-6}, layers=rows)
    heads = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"], "scale": s["dim"] ** -0.5}
    full = dict(heads, conv=4, softcap=30.0, rot={"dims": s["dim"], "base": 5e5, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})
    left = dict(heads, buckets=s["buckets"], bias_max=s["far"], mask={"size": s["window"], "keep_first": s["keep_first"]})
    right = {"heads": s["space_heads"], "groups": s["groups"], "state": s["state"], "vdim": s["space_vdim"], "conv": 4, "norm_groups": s["groups"]}
    pair, attention = {"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": dense}, {"type": "attention", "mixer": full, "mlp": dense}
    return dict(out, architecture="Kukulorn", logit_softcap=30.0, layers=[pair, pair, attention, pair, attention], loop={"start": 0, "stop": 3, "times": 2})


def depth(model: str, layers: int) -> int:
    return layers if SIZES[model]["design"] == "qwen2" else 8


class Weights:
    """A model's tensors by their checkpoint names, each drawn from a generator of its own, so that they can be had in any
    order.  The law is that of an initialised model: matrices that keep a row's size, output projections smaller by the
    root of the depth, norm weights near one, decays and step sizes spread over the range that such models start from."""

    def __init__(self, model: str, layers: int, dtype: str, shapes=None) -> None:
        self.model, self.layers, self.dtype, self.shapes = model, depth(model, layers), DTYPES[dtype], shapes

    def names(self):
        return self.shapes.keys()

    def __contains__(self, name: str) -> bool:
        return name in self.shapes

    def shape(self, name: str):
        return self.shapes[name]

    def tensor(self, name: str) -> torch.Tensor:
        return self.draw(name, self.shapes[name])

    def draw(self, name: str, shape) -> torch.Tensor:
        generator = torch.Generator(device=DEVICE)
        generator.manual_seed(zlib.crc32(f"{self.model} {name}".encode()))
        last = name.rsplit(".", 1)[-1]
        plain = torch.randn(tuple(shape), generator=generator, device=DEVICE)
        small = 0.02 * plain
        if last in ("A_log", "dt_bias", "w0"):
            share = torch.rand(tuple(shape), generator=generator, device=DEVICE)
            if last == "A_log":
                value = torch.log(1.0 + 15.0 * share)
            elif last == "dt_bias":  # softplus of it is spread over 0.001 .. 0.1
                step = torch.exp(math.log(0.001) + share * math.log(100.0))
                value = step + torch.log(-torch.expm1(-step))
            else:
                value = -6.0 * share
        elif last == "embed" or "embed_tokens" in name:
            value = plain * {"qwen2": 0.02, "tiverax": 0.02, "gosulorn": 0.1, "kedanex": 1.0, "kukulorn": 0.1}[SIZES[self.model]["design"]]
            if "experts" in SIZES[self.model]:  # experts follow the tokens, as trained routers have it: some channels speak up and the router listens to them
                value[:, :shape[1] // 32] *= 6.0
        elif last in ("norm1b", "norm2b") or name.endswith(("mix.left.out", "mix.right.out")):
            value = (0.15 if last in ("norm1b", "norm2b") else 0.3) + small  # norms of a sub-layer's output
        elif "norm" in name or last in ("D",):
            value = 1.0 + small
        elif ".hc" in name:
            value = small + {"in": 1.0 / shape[0], "out": 1.0}[last] if last != "mix" else small + torch.eye(shape[0], device=DEVICE)
        elif last == "act":
            value = small + torch.tensor([1.0, 1.0, 1.0, 0.0], device=DEVICE) / 3.0
        elif last == "conv":
            value = 0.3 * plain
        elif last == "router":
            value = plain * (0.1 * shape[1] ** -0.5)
            value[:, :shape[1] // 32] = plain[:, :shape[1] // 32] * (0.4 * (shape[1] // 32) ** -0.5)
        elif last == "rel":
            value = 0.5 * plain
        elif len(shape) == 1:
            value = 0.1 * plain  # biases
        elif last in ("o", "down") or name.endswith(("o_proj.weight", "down_proj.weight")):
            value = plain * (shape[1] ** -0.5 * (2 * self.layers) ** -0.5)
        else:
            value = plain * shape[1] ** -0.5
        return value.to(self.dtype)


_loaded = {}  # the model that the last case used: a serving program loads its weights once


def loaded_model(model: str, layers: int, dtype: str) -> DecoderModel:
    key = (model, layers, dtype)
    if key not in _loaded:
        _loaded.clear()
        config = config_from_dict(model_config(model, layers))
        built = DecoderModel(get_architecture(config.architecture).make_spec(config, 32768))
        shapes = {}
        for _part, _attr, param, names in expected_names(built.all_parts()):
            if param.alias_of is None:
                shapes.update(zip(names, (tuple(s) for s in param.source_shapes)))
        bind(built, Weights(model, layers, dtype, shapes), DTYPES[dtype], DEVICE)
        load_ops(DEVICE).prepare(built, DTYPES[dtype])
        _loaded[key] = built
    return _loaded[key]


# ----------------------------------------------------------------------------------------------------------------------
# cases
# ----------------------------------------------------------------------------------------------------------------------
def step_case(model, dtype="bfloat16", layers=8, decodes=0, low=0, high=0, portions=0, shortest=0, longest=0, behind=0, **more) -> dict:
    return dict(more, model=model, dtype=dtype, layers=depth(model, layers), decodes=decodes, low=low, high=high, portions=portions, shortest=shortest, longest=longest, behind=behind)


def listed():
    return [
        # one user's chat with the small model: every launch counts; all 28 layers, as nothing else hides the host
        step_case("qwen2-1.5b", layers=28, decodes=1, low=391, high=391, name="decode-1-qwen2-1.5b"),
        # the engine's headline: eight requests behind 4,096 tokens each
        step_case("qwen2-7b", decodes=8, low=4096, high=4096, name="decode-8-qwen2-7b"),
        # a busy server between prompts: an odd number of requests, each at another place of its answer
        step_case("qwen2-7b", decodes=57, low=65, high=1500, name="decode-57-qwen2-7b"),
        # a busy server's usual step: decoding requests beside a 512-token portion of a longer prompt and a short new one
        step_case("qwen2-7b", decodes=23, low=100, high=2000, portions=2, shortest=301, longest=512, name="step-qwen2-7b"),
        # one prompt read at once (retrieval, a long question)
        step_case("qwen2-7b", portions=1, shortest=2048, longest=2048, name="prompt-qwen2-7b"),
        # the true 32-bit path: a small serving step
        step_case("qwen2-1.5b", dtype="float32", decodes=5, low=100, high=900, portions=1, shortest=611, longest=611, name="float32-step-qwen2-1.5b"),
        # drawing the tokens of a busy server's step
        dict(name="sample-48", rows=48, vocab=152064, temperature=0.8, top_p=0.9, top_k=0, greedy=6),
        # prompts through routed experts and attention over a latent
        step_case("tiverax-4k", portions=2, shortest=1000, longest=1500, name="prompts-tiverax-4k"),
        # prompts of unequal length through delta rules and window attention
        step_case("gosulorn-2k", portions=3, shortest=400, longest=1300, name="prompts-gosulorn-2k"),
        # a serving step through the generalized delta rule, gated recurrences and experts
        step_case("kedanex-2k", decodes=12, low=50, high=1500, portions=1, shortest=1024, longest=1024, name="step-kedanex-2k"),
        # a long prompt through state spaces, windows with kept tokens and capped attention
        step_case("kukulorn-4k", portions=1, shortest=4001, longest=4001, name="prompt-kukulorn-4k"),
        # decoding through experts and latents: the weights of the experts that were hit, and many small kernels
        step_case("tiverax-4k", decodes=16, low=100, high=3000, name="decode-16-tiverax-4k"),
    ]


def _spread(rng: random.Random, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random) -> dict:
    """One more case of the same ranges."""
    most = max(_size(c) for c in listed())
    while True:
        if rng.random() < 0.1:
            return dict(rows=_spread(rng, 1, 64), vocab=rng.choice((32000, 151936, 152064)), temperature=rng.choice((0.6, 0.8, 1.0)), top_p=rng.choice((1.0, 0.95, 0.9, 0.5)),
                        top_k=rng.choice((0, 0, 20, 50)), greedy=rng.choice((0, 2, 6)))
        model = rng.choice(sorted(SIZES))
        dtype = "float32" if rng.random() < 0.15 and model in ("qwen2-1.5b", "gosulorn-2k", "kukulorn-2k") else "bfloat16"
        case = step_case(model, dtype, layers=rng.choice((4, 8)))
        kind = rng.choice(("decode", "prompts", "both"))
        if kind != "prompts":
            case["decodes"] = _spread(rng, 1, 64)
            bounds = sorted(_spread(rng, 16, 4096) for _ in range(2))
            case["low"], case["high"] = bounds
        if kind != "decode":
            case["portions"] = rng.choice((1, 1, 2, 3))
            bounds = sorted(_spread(rng, 16, 4096 // case["portions"]) for _ in range(2))
            case["shortest"], case["longest"] = bounds
            case["behind"] = rng.choice((0, 0, 0, 512, 1000))
        tokens = sum(contexts(case)) + sum(prompts(case)) + case["portions"] * case["behind"]
        if _size(case) <= 0.8 * most and tokens <= 50000 and tokens * max(contexts(case) + prompts(case)) <= 1.2e8:
            return case


def _between(low: int, high: int, count: int):
    """``count`` whole numbers from ``low`` to ``high``, evenly over the logarithm, in no order."""
    if count <= 0:
        return []
    out = [int(round(low * (high / low) ** (i / max(1, count - 1)))) for i in range(count)] if count > 1 else [high]
    random.Random(count).shuffle(out)
    return out


def contexts(case):
    return _between(case["low"], case["high"], case["decodes"])


def prompts(case):
    return _between(case["shortest"], case["longest"], case["portions"])


def token_ids(case, seed: int):
    """For every decoding request its context and the token it brings, for every portion what was read before it and its own
    tokens: lists of token ids, uniform over the vocabulary."""
    vocab = SIZES[case["model"]]["vocab"]
    lengths = [n + 1 for n in contexts(case)] + [case["behind"] + n for n in prompts(case)]
    generator = torch.Generator().manual_seed(int(seed))
    return [torch.randint(0, vocab, (n,), generator=generator).tolist() for n in lengths]


# ----------------------------------------------------------------------------------------------------------------------
# a user's program
# ----------------------------------------------------------------------------------------------------------------------
class Step:
    """A runner with its cache, the requests that decode, and the portions of prompts that one pass reads."""

    def __init__(self, runner, cache, decodes, portions) -> None:
        self.runner, self.cache, self.decodes, self.portions = runner, cache, decodes, portions


class Draws:
    def __init__(self, sampler, logits, params) -> None:
        self.sampler, self.logits, self.params = sampler, logits, params
        self.ids = [f"request {r}" for r in range(len(params))]
        self.generated = [7 * r + 1 for r in range(len(params))]


def prepare(case, seed):
    if "rows" in case:
        generator = torch.Generator(device=DEVICE)
        generator.manual_seed(int(seed))
        logits = 3.0 * torch.randn((case["rows"], case["vocab"]), generator=generator, device=DEVICE)
        params = [SamplingParams(temperature=0.0) if case["greedy"] and r % case["greedy"] == 0
                  else SamplingParams(temperature=case["temperature"], top_p=case["top_p"], top_k=case["top_k"], seed=int(seed) + r) for r in range(case["rows"])]
        return Draws(Sampler(load_ops(DEVICE), DEVICE, seed=int(seed)), logits, params)

    model, dtype = loaded_model(case["model"], case["layers"], case["dtype"]), DTYPES[case["dtype"]]
    ids = token_ids(case, seed)
    tokens = case["decodes"] + sum(prompts(case))
    sequences = len(ids)
    slots = 1 << (sequences - 1).bit_length()
    pages = sum((len(row) + PAGE - 1) // PAGE for row in ids) + 2
    longest = max(len(row) for row in ids)
    cache = CacheManager(model.cache_needs(), PAGE, pages, slots, dtype, DEVICE, max_model_len=longest + PAGE, scatter_pages=True)
    runner = ModelRunner(model, cache, load_ops(DEVICE), dtype, DEVICE, max_num_tokens=max(tokens, min(READ_CHUNK, sum(len(row) for row in ids))), max_num_seqs=slots,
                         enable_graphs=case["portions"] == 0)
    if case["portions"] == 0:
        runner.capture_decode_graphs([slots])

    # what earlier steps have left in the cache
    held = contexts(case) + [case["behind"]] * case["portions"]
    kept, step, room = [], [], runner.max_num_tokens
    for row, length in zip(ids, held):
        seq = cache.new_sequence() if length else None
        kept.append(seq)
        at = 0
        while at < length:
            count = min(length - at, room)
            cache.append(seq, at, count)
            step.append(StepEntry(seq, row[at:at + count], at, []))
            at, room = at + count, room - count
            if room == 0 or at < length:
                _read(runner, cache, step)
                step, room = [], runner.max_num_tokens
    _read(runner, cache, step)
    decodes = [(seq, row[-1:], len(row) - 1) for seq, row in zip(kept, ids[:case["decodes"]])]
    for seq, _token, start in decodes:
        cache.append(seq, start, 1)
    portions = []
    for seq, row in zip(kept[case["decodes"]:], ids[case["decodes"]:]):
        portions.append((seq, row[case["behind"]:]))
        if seq is not None:
            cache.append(seq, case["behind"], len(row) - case["behind"])
    return Step(runner, cache, [StepEntry(seq, token, start, [0]) for seq, token, start in decodes],
                [(seq, row, case["behind"]) for seq, row in portions])


def _read(runner, cache, entries) -> None:
    if entries:
        runner.step(entries)
        for entry in entries:
            cache.release_behind_window(entry.seq, entry.start + len(entry.token_ids))


def run(state):
    if isinstance(state, Draws):
        return {"tokens": state.sampler.sample(state.logits, state.params, state.ids, state.generated)}
    entries, new = list(state.decodes), []
    for seq, row, start in state.portions:
        if seq is None:  # a prompt's first portion: the request gets its slot and pages now
            seq = state.cache.new_sequence()
            state.cache.append(seq, start, len(row))
            new.append(seq)
        entries.append(StepEntry(seq, row, start, [len(row) - 1]))
    logits = state.runner.step(entries)
    for seq in new:
        state.cache.free_sequence(seq)
    return {"logits": logits}


# ----------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------------------------------
def _layers(case):
    """Per run of a layer: (numbers in its matrices, whether they were counted before, experts, experts a token uses, numbers in one
    expert's matrices, heads, head size of keys and values together, numbers a token leaves in the cache (0: borrowed), window,
    operations of the recurrence per token, numbers of state)."""
    s = SIZES[case["model"]]
    w, out = s["width"], []
    if s["design"] == "qwen2":
        n = w * (2 * s["heads"] + 2 * s["kv_heads"]) * s["dim"] + 3 * w * s["ff"]
        return [(n, False, 0, 0, 0, s["heads"], 2 * s["dim"], 2 * s["kv_heads"] * s["dim"], 0, 0, 0)] * case["layers"]
    dense = 3 * w * s["ff"]
    if s["design"] == "tiverax":
        expert = 3 * w * s["expert_ff"]
        for i in range(8):
            n = w * s["heads"] * (s["dim"] + s["rot_dim"]) + 2 * w * s["heads"] * s["vdim"] + s["heads"] * (s["dim"] + s["vdim"]) * s["kv_rank"]
            n += w * (s["kv_rank"] + s["rot_dim"]) if i % 4 < 2 else 0
            moe = i % 2 == 1
            out.append((n + (3 * w * s["shared_ff"] + w * s["experts"] if moe else dense), False, s["experts"] if moe else 0, s["top"], expert, s["heads"],
                        2 * s["kv_rank"] + s["rot_dim"], s["kv_rank"] + s["rot_dim"] if i % 4 < 2 else 0, 0, 0, 0))
        return out
    d = s["dim"]
    attention = w * (2 * s["heads"] + 2 * s["kv_heads"]) * d
    kv = 2 * s["kv_heads"] * d
    if s["design"] == "gosulorn":
        right = w * (4 * s["right_heads"] * d + s["right_heads"] + 2 * s["rank"]) + 2 * s["rank"] * s["right_heads"] * d
        gla = w * (2 * s["gla_heads"] * d + 3 * s["gla_heads"] * s["gla_vdim"] + s["rank"]) + s["rank"] * s["gla_heads"] * d
        delta = w * (2 * s["delta_kv_heads"] * d + 3 * s["delta_heads"] * d + 2 * s["delta_heads"])
        kinds = [(attention + right + dense, False, 0, 0, 0, s["heads"], 2 * d, kv, s["window"], 7 * s["right_heads"] * d * d, s["right_heads"] * d * d),
                 (gla + dense, False, 0, 0, 0, 0, 0, 0, 0, 5 * s["gla_heads"] * d * s["gla_vdim"], s["gla_heads"] * d * s["gla_vdim"]),
                 (delta + dense, False, 0, 0, 0, 0, 0, 0, 0, 7 * s["delta_heads"] * d * d, s["delta_heads"] * d * d)]
        return [kinds[i] for i in (0, 1, 0, 2) * 2]
    if s["design"] == "kedanex":
        e = s["delta_dim"]
        delta = 6 * w * s["delta_heads"] * e + s["rank"] * (w + s["delta_heads"] * e)
        scan = 9 * s["delta_heads"] * e * e
        expert = 3 * w * s["expert_ff"]
        moe = (False, s["experts"], s["top"], expert)
        router = w * s["experts"]
        four = [(delta + 2 * w * s["ff"], False, 0, 0, 0, 0, 0, 0, 0, scan, s["delta_heads"] * e * e), (4 * w * s["gru_width"] + router, *moe, 0, 0, 0, 0, 4 * s["gru_width"], s["gru_width"]),
                (attention - w * s["kv_heads"] * d + router, *moe, s["heads"], 2 * d, kv, s["window"], 0, 0), (delta + router, *moe, 0, 0, 0, 0, scan, s["delta_heads"] * e * e)]
        rows = four * 2
        rows[7] = (rows[7][0], True) + rows[7][2:]
        return rows
    inner, gn = s["space_heads"] * s["space_vdim"], s["groups"] * s["state"]
    space = w * (3 * inner + 2 * gn + s["space_heads"])
    n = s["space_heads"] * s["state"] * s["space_vdim"]
    pair = (attention + w * s["heads"] + space + dense, False, 0, 0, 0, s["heads"], 2 * d, kv, s["window"], 5 * n, n)
    full = (attention + w * s["heads"] * d + dense, False, 0, 0, 0, s["heads"], 2 * d, kv, 0, 0, 0)
    again = [row[:1] + (True,) + row[2:] for row in (pair, pair, full)]
    first = (pair[0] + 2 * w * w,) + pair[1:]
    return [first, pair, full] + [(again[0][0] + 2 * w * w,) + again[0][1:]] + again[1:] + [pair, full]


def work(case):
    if "rows" in case:
        return {"bytes": 4 * case["rows"] * case["vocab"] + 4 * case["rows"], "flops": 3 * case["rows"] * case["vocab"]}
    s = SIZES[case["model"]]
    size = 4 if case["dtype"] == "float32" else 2
    spans = [(n, 1) for n in contexts(case)] + [(case["behind"], n) for n in prompts(case)]  # (tokens before, tokens of the step)
    tokens, wanted = sum(n for _, n in spans), len(spans)
    head = s["vocab"] * s["width"]
    nbytes, flops = head * size + tokens * s["width"] * size + wanted * s["vocab"] * 4, 2 * wanted * head
    for n, counted, experts, top, expert, heads, dims, kv, window, scan, state in _layers(case):
        hit = min(experts, tokens * top)
        nbytes += 0 if counted else (n + hit * expert) * size
        flops += 2 * tokens * (n + (top * expert if experts else 0)) + tokens * scan
        nbytes += 8 * state * len(spans)
        for before, own in spans:
            if window:
                pairs = sum(min(window, before + i + 1) for i in range(own)) if own < 64 else own * min(window, before + own) - (min(window, own) ** 2 / 2 if before < window else 0)
                seen = min(before, window)
            else:
                pairs, seen = own * before + own * (own + 1) / 2, before
            flops += 2 * pairs * heads * dims
            nbytes += (seen + own) * kv * size
    return {"bytes": nbytes, "flops": flops}


def _size(case) -> float:
    """A case's cost in seconds, roughly: a step cannot be faster than its bytes or its operations allow."""
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / (1e14 if case.get("dtype") == "float32" else 1e15))


def tolerance(case):
    if "rows" in case:
        return "exact"  # the draw is defined bit for bit by the logits, the options and the request's seed
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    if SIZES[case["model"]]["design"] in ("tiverax", "kedanex"):
        return {"rel": 0.02, "max": 0.6}  # a token near a border between two experts may go to the other one
    return {"rel": 0.03 if SIZES[case["model"]]["design"] == "gosulorn" else 0.02, "max": 0.25}


# ----------------------------------------------------------------------------------------------------------------------
# the same logits in 64 bits, written out plainly: all sequences side by side [B, n, ...], padded at their ends, no cache
# ----------------------------------------------------------------------------------------------------------------------
def silu(z):
    return z * torch.sigmoid(z)


def over_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def rotate(x, freqs, magnitude=1.0, pairs=False):
    """``x`` [B, n, heads, d]: channels ``i`` and ``i + half`` (or ``2 i`` and ``2 i + 1``) of the first ``2 len(freqs)`` are turned."""
    half = len(freqs)
    angle = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * torch.tensor(freqs, dtype=torch.float64, device=x.device)
    cos, sin = (angle.cos() * magnitude)[:, None, :], (angle.sin() * magnitude)[:, None, :]
    out = x.clone()
    at, to = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if pairs else (slice(0, half), slice(half, 2 * half))
    u, v = x[..., at], x[..., to]
    out[..., at], out[..., to] = u * cos - v * sin, v * cos + u * sin
    return out


def causal_conv(u, weight):
    taps = weight.shape[1]
    out = u * weight[:, -1]
    for back in range(1, taps):
        out[:, back:] += u[:, :-back] * weight[:, taps - 1 - back]
    return out


def attend(q, k, v, scale, window=0, keep=0, bias=None, cap=0.0, silent=False):
    """Causal softmax attention; ``q`` [B, n, heads, d], ``k`` and ``v`` [B, n, groups, ...].  ``bias`` [heads, n] by distance; ``silent``: one
    more key of score 0 without a value."""
    batch, n, heads, _ = q.shape
    group = heads // k.shape[2]
    out = q.new_zeros(batch, n, heads, v.shape[-1])
    place = torch.arange(n, device=q.device)
    for b in range(batch):
        keys = k[b].permute(1, 2, 0).contiguous()  # [groups, d, n]
        values = v[b].permute(1, 0, 2).contiguous()
        for lo in range(0, n, 512):
            hi = min(n, lo + 512)
            rows = q[b, lo:hi].permute(1, 0, 2).reshape(k.shape[2], group * (hi - lo), -1).contiguous()
            scores = (torch.bmm(rows, keys[:, :, :hi].contiguous()) * scale).reshape(heads, hi - lo, hi)
            distance = place[lo:hi, None] - place[None, :hi]
            if cap:
                scores = cap * torch.tanh(scores / cap)
            if bias is not None:
                scores = scores + bias[:, distance.clamp(min=0)]
            hidden = distance < 0
            if window:
                hidden = hidden | ((distance >= window) & (place[None, :hi] >= keep))
            scores = scores.masked_fill(hidden, float("-inf"))
            if silent:
                scores = torch.cat([scores, scores.new_zeros(heads, hi - lo, 1)], dim=-1)
            weights = torch.softmax(scores, dim=-1)[..., :hi].reshape(k.shape[2], group * (hi - lo), hi)
            out[b, lo:hi] = torch.bmm(weights, values[:, :hi].contiguous()).reshape(heads, hi - lo, -1).permute(1, 0, 2)
    return out


class Plain:
    """The model of a case in 64 bits.  ``w(name, *shape)`` is the tensor as the run holds it."""

    def __init__(self, case) -> None:
        self.case, self.s = case, SIZES[case["model"]]
        self.config = model_config(case["model"], case["layers"])
        self.weights = Weights(case["model"], case["layers"], case["dtype"])
        self.eps = self.config["rms_norm_eps"] if "rms_norm_eps" in self.config else self.config["norm"]["eps"]

    def w(self, name, *shape):
        return self.weights.draw(name, shape).double()

    def product(self, x, name, rows):
        return x @ self.w(name, rows, x.shape[-1]).T

    def norm(self, x, name):
        return over_rms(x, self.eps) * self.w(name, x.shape[-1])

    def logits(self, ids, rows):
        """``ids`` [B, n]; ``rows``: per sequence the place whose logits are wanted."""
        return getattr(self, self.s["design"])(ids, (torch.arange(len(rows), device=ids.device), torch.tensor(rows, device=ids.device)))

    # -- Qwen2 ----------------------------------------------------------------------------------------------------------
    def qwen2(self, ids, rows):
        s = self.s
        table = self.w("model.embed_tokens.weight", s["vocab"], s["width"])
        x = table[ids]
        if not s["tied"]:
            del table
        freqs = [1e6 ** (-2.0 * i / s["dim"]) for i in range(s["dim"] // 2)]
        for layer in range(self.case["layers"]):
            p = f"model.layers.{layer}."
            h = self.norm(x, p + "input_layernorm.weight")
            q, k, v = (self.product(h, f"{p}self_attn.{name}_proj.weight", n * s["dim"]).add_(self.w(f"{p}self_attn.{name}_proj.bias", n * s["dim"])).unflatten(-1, (n, s["dim"]))
                       for name, n in (("q", s["heads"]), ("k", s["kv_heads"]), ("v", s["kv_heads"])))
            y = attend(rotate(q, freqs), rotate(k, freqs), v, s["dim"] ** -0.5)
            x = x + self.product(y.flatten(2), p + "self_attn.o_proj.weight", s["width"])
            h = self.norm(x, p + "post_attention_layernorm.weight")
            x = x + self.product(silu(self.product(h, p + "mlp.gate_proj.weight", s["ff"])) * self.product(h, p + "mlp.up_proj.weight", s["ff"]), p + "mlp.down_proj.weight", s["width"])
        x = self.norm(x[rows], "model.norm.weight")
        return x @ (table if s["tied"] else self.w("lm_head.weight", s["vocab"], s["width"])).T

    # -- shared by the other designs ---------------------------------------------------------------------------------------
    def gated(self, h, p, ff, activation=silu):
        return self.product(activation(self.product(h, p + "gate", ff)) * self.product(h, p + "up", ff), p + "down", self.s["width"])

    def experts(self, h, p, choose, scale_input):
        flat = h.reshape(-1, h.shape[-1])
        index, weight = choose(self.product(flat, p + "router", self.s["experts"]))
        out = torch.zeros_like(flat)
        for e in range(self.s["experts"]):
            row, place = (index == e).nonzero(as_tuple=True)
            share = weight[row, place][:, None]
            y = self.gated(flat[row] * share if scale_input else flat[row], f"{p}e{e}.", self.s["expert_ff"])
            out[row] += y if scale_input else share * y
        return out.reshape(h.shape)

    # -- Tiverax --------------------------------------------------------------------------------------------------------
    def tiverax(self, ids, rows):
        s, width = self.s, self.s["width"]
        rot, dim, vdim, heads, rank = s["rot_dim"], s["dim"], s["vdim"], s["heads"], s["kv_rank"]
        x = self.w("embed", s["vocab"], width)[ids] * width ** 0.5
        freqs = [1e6 ** (-2.0 * i / rot) for i in range(rot // 2)]
        turn = [rot * math.log(4096 / (2.0 * math.pi * t)) / (2.0 * math.log(1e6)) for t in (32.0, 1.0)]
        lo, hi = max(math.floor(turn[0]), 0), min(math.ceil(turn[1]), rot - 1)
        ramp = [min(1.0, max(0.0, (i - lo) / max(hi - lo, 0.001))) for i in range(rot // 2)]
        freqs = [f / 4.0 * r + f * (1.0 - r) for f, r in zip(freqs, ramp)]
        magnitude = 0.1 * math.log(4.0) + 1.0

        def choose(z):
            score = torch.sigmoid(z)
            index = score.topk(s["top"], dim=-1).indices
            return index, score.gather(-1, index)

        kept = {}
        for i, layer in enumerate(self.config["layers"]):
            p, source = f"l{i}.", layer["mixer"].get("kv_from", i)
            h = self.norm(x, p + "norm1")
            if source == i:
                down = self.product(h, p + "mix.dkv", rank + rot)
                kept[i] = (over_rms(down[..., :rank], self.eps) * self.w(p + "mix.dkv.norm", rank), rotate(down[:, :, None, rank:], freqs, magnitude, pairs=True))
            latent, shared = kept[source]
            q = self.product(h, p + "mix.q", heads * (dim + rot)).unflatten(-1, (heads, dim + rot))
            q = torch.cat([q[..., :dim], rotate(q[..., dim:], freqs, magnitude, pairs=True)], dim=-1)
            k = torch.cat([self.product(latent, p + "mix.uk", heads * dim).unflatten(-1, (heads, dim)), shared.expand(-1, -1, heads, -1)], dim=-1)
            v = self.product(latent, p + "mix.uv", heads * vdim).unflatten(-1, (heads, vdim))
            y = attend(q, k, v, (dim + rot) ** -0.5).flatten(2) * torch.sigmoid(self.product(h, p + "mix.g", heads * vdim))
            y = self.product(y, p + "mix.o", width)
            if layer["mlp"]["kind"] == "moe":
                x = x + y + self.experts(h, p + "mlp.", choose, True) + self.gated(h, p + "mlp.shared.", s["shared_ff"])
            else:
                x = x + y + self.gated(h, p + "mlp.", s["ff"])
        return self.product(self.norm(x[rows], "final.norm"), "head", s["vocab"])

    # -- Gosulorn -------------------------------------------------------------------------------------------------------
    def gosulorn(self, ids, rows):
        s, width = self.s, self.s["width"]
        table = self.w("embed", s["vocab"], width)
        xs = [table[ids] for _ in range(s["streams"])]

        def layer_norm(x, name):
            x = x - x.mean(-1, keepdim=True)
            return over_rms(x, self.eps) * self.w(name, width)

        for i, layer in enumerate(self.config["layers"]):
            p = f"l{i}."
            for number in (1, 2):
                into, out, mix = (self.w(f"{p}hc{number}.{name}", *shape) for name, shape in (("in", (4,)), ("out", (4,)), ("mix", (4, 4))))
                h = layer_norm(sum(into[a] * xs[a] for a in range(4)), f"{p}norm{number}")
                y = getattr(self, "gosulorn_" + layer["type"])(h, p + "mix.", layer["mixer"]) if number == 1 else self.gated(
                    h, p + "mlp.", s["ff"], lambda z: torch.nn.functional.gelu(z, approximate="tanh"))
                xs = [sum(mix[a, to] * xs[a] for a in range(4)) + out[to] * y for to in range(4)]
        return layer_norm(sum(xs)[rows], "final.norm") @ table.T

    def conv_heads(self, h, name, heads, dim):
        return causal_conv(self.product(h, name, heads * dim), self.w(name + ".conv", heads * dim, 4)).unflatten(-1, (heads, dim))

    def delta_rule(self, h, p, c, decay):
        heads, kv, dim = c["heads"], c["kv_heads"], c["dim"]
        q = (unit(silu(self.conv_heads(h, p + "q", kv, dim))) * dim ** -0.5).repeat_interleave(heads // kv, dim=2)
        k = unit(silu(self.conv_heads(h, p + "k", kv, dim))).repeat_interleave(heads // kv, dim=2)
        v = silu(self.conv_heads(h, p + "v", heads, c["vdim"]))
        beta = torch.sigmoid(self.product(h, p + "b", heads))
        state, out = h.new_zeros(h.shape[0], heads, dim, c["vdim"]), torch.zeros_like(v)
        for t in range(h.shape[1]):
            state = state * decay[:, t, :, :, None]
            u = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None, :], state)[:, :, 0])
            state.add_(k[:, t, :, :, None] * u[:, :, None, :])
            out[:, t] = torch.matmul(q[:, t, :, None, :], state)[:, :, 0]
        return over_rms(out, self.eps) * self.w(p + "norm", c["vdim"])

    def gosulorn_delta(self, h, p, c):
        heads = c["heads"]
        step = torch.nn.functional.softplus(self.product(h, p + "a", heads) + self.w(p + "dt_bias", heads))
        decay = torch.exp(-torch.exp(self.w(p + "A_log", heads)) * step)[..., None].expand(-1, -1, -1, c["dim"])
        o = self.delta_rule(h, p, c, decay) * silu(self.product(h, p + "g", heads * c["vdim"])).unflatten(-1, (heads, -1))
        return self.product(o.flatten(2), p + "o", self.s["width"])

    def gosulorn_parallel(self, h, p, c):
        s, left, right = self.s, c["left"], c["right"]
        d, heads = left["dim"], right["heads"]

        def projected(name, n):
            y = self.product(h, f"{p}left.{name}", n * d) + self.w(f"{p}left.{name}.b", n * d)
            return causal_conv(y, self.w(f"{p}left.{name}.conv", n * d, 4)).unflatten(-1, (n, d))

        freqs = [1e6 ** (-2.0 * i / (d // 2)) / 4.0 for i in range(d // 4)]
        q, k, v = projected("q", s["heads"]), projected("k", s["kv_heads"]), projected("v", s["kv_heads"])
        y = attend(rotate(q, freqs), rotate(k, freqs), v, d ** -0.5, window=s["window"]).flatten(2)
        y = self.product(y, p + "left.o", s["width"]) + self.w(p + "left.o.b", s["width"])
        r = p + "right."
        inner = heads * right["dim"]
        step = torch.nn.functional.softplus(self.product(self.product(h, r + "a1", s["rank"]), r + "a2", inner) + self.w(r + "dt_bias", inner)).unflatten(-1, (heads, -1))
        decay = torch.exp(-torch.exp(self.w(r + "A_log", heads))[:, None] * step)
        gate = torch.sigmoid(self.product(self.product(h, r + "g1", s["rank"]), r + "g2", inner)).unflatten(-1, (heads, -1))
        o = (self.delta_rule(h, r, right, decay) * gate).flatten(2)
        return c["left_scale"] * y + c["right_scale"] * self.product(o, r + "o", s["width"])

    def gosulorn_gla(self, h, p, c):
        heads, dim, vdim = c["heads"], c["dim"], c["vdim"]
        q = self.product(h, p + "q", heads * dim).unflatten(-1, (heads, dim)) * dim ** -0.5
        k = self.product(h, p + "k", heads * dim).unflatten(-1, (heads, dim))
        v = self.product(h, p + "v", heads * vdim).unflatten(-1, (heads, vdim))
        z = self.product(self.product(h, p + "a1", c["a1_rank"]), p + "a2", heads * dim) + self.w(p + "a2.b", heads * dim)
        decay = (torch.sigmoid(z) ** (1.0 / c["tau"])).unflatten(-1, (heads, dim))
        state, out = h.new_zeros(h.shape[0], heads, dim, vdim), torch.zeros_like(v)
        for t in range(h.shape[1]):
            state = state * decay[:, t, :, :, None] + k[:, t, :, :, None] * v[:, t, :, None, :]
            out[:, t] = torch.matmul(q[:, t, :, None, :], state)[:, :, 0]
        o = (over_rms(out, self.eps) * self.w(p + "norm", vdim)).flatten(2) * silu(self.product(h, p + "g", heads * vdim))
        return self.product(o, p + "o", self.s["width"])

    # -- Kedanex --------------------------------------------------------------------------------------------------------
    def kedanex(self, ids, rows):
        s = self.s

        def choose(z):
            value, index = z.topk(s["top"], dim=-1)
            return index, torch.softmax(value, dim=-1)

        x = self.w("embed", s["vocab"], s["width"])[ids]
        for i, layer in enumerate(self.config["layers"]):
            p = f"l{layer.get('weights_of', i)}."
            x = x + self.norm(getattr(self, "kedanex_" + layer["type"])(self.norm(x, p + "norm1"), p + "mix.", layer["mixer"]), p + "norm1b")
            h = self.norm(x, p + "norm2")
            if layer["mlp"]["kind"] == "moe":
                y = self.experts(h, p + "mlp.", choose, False)
            else:
                z, c = self.product(h, p + "mlp.up", s["ff"]), self.w(p + "mlp.act", 4)
                y = self.product(c[0] * over_rms(z, self.eps) + c[1] * over_rms(z ** 2, self.eps) + c[2] * over_rms(z ** 3, self.eps) + c[3], p + "mlp.down", s["width"])
            x = x + self.norm(y, p + "norm2b")
        return self.product(self.norm(x[rows], "final.norm"), "head", s["vocab"])

    def kedanex_general_delta(self, h, p, c):
        heads, dim = c["heads"], c["dim"]
        inner = heads * dim
        r, k, v = (self.product(h, p + name, inner).unflatten(-1, (heads, dim)) for name in ("r", "k", "v"))
        removal = torch.sigmoid(self.product(h, p + "a", inner) + self.w(p + "a.b", inner)).unflatten(-1, (heads, dim))
        z = self.product(torch.tanh(self.product(h, p + "w1", c["w1_rank"])), p + "w2", inner) + self.w(p + "w0", inner)
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(z)).unflatten(-1, (heads, dim))
        u = unit(k)
        taken = removal * u
        state, out = h.new_zeros(h.shape[0], heads, dim, dim), torch.zeros_like(v)
        for t in range(h.shape[1]):
            seen = torch.matmul(u[:, t, :, None, :], state)
            state = state * decay[:, t, :, :, None] - taken[:, t, :, :, None] * seen + k[:, t, :, :, None] * v[:, t, :, None, :]
            out[:, t] = torch.matmul(r[:, t, :, None, :], state)[:, :, 0]
        o = over_rms(out, self.eps).flatten(2) * self.w(p + "norm", inner) * torch.sigmoid(self.product(h, p + "g", inner))
        return self.product(o, p + "o", self.s["width"])

    def kedanex_mingru(self, h, p, c):
        n = c["width"]
        z = torch.sigmoid(self.product(h, p + "z", n) + self.w(p + "z.b", n))
        u = self.product(h, p + "x", n) + self.w(p + "x.b", n)
        fresh = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
        state, out = h.new_zeros(h.shape[0], n), torch.zeros_like(z)
        for t in range(h.shape[1]):
            state = (1.0 - z[:, t]) * state + fresh[:, t]
            out[:, t] = state
        return self.product(out * silu(self.product(h, p + "g", n)), p + "o", self.s["width"])

    def kedanex_attention(self, h, p, c):
        d = c["dim"]
        q, v = (self.product(h, p + name, n * d).unflatten(-1, (n, d)) for name, n in (("q", c["heads"]), ("k", c["kv_heads"])))
        freqs = [1e6 ** (-2.0 * i / d) for i in range(d // 2)]
        y = attend(over_rms(rotate(q, freqs), self.eps), over_rms(rotate(v, freqs), self.eps), v, d ** -0.5, window=c["mask"]["size"], silent=True)
        return self.product(y.flatten(2), p + "o", self.s["width"])

    # -- Kukulorn -------------------------------------------------------------------------------------------------------
    def kukulorn(self, ids, rows):
        s, loop = self.s, self.config["loop"]
        table = self.w("embed", s["vocab"], s["width"])
        x = start = table[ids]
        order = [(i, i == loop["start"]) for _ in range(loop["times"]) for i in range(loop["start"], loop["stop"])] + [(i, False) for i in range(loop["stop"], 5)]
        for i, begins_pass in order:
            layer, p = self.config["layers"][i], f"l{i}."
            if begins_pass:
                x = self.product(torch.cat([x, start], dim=-1), "loop.in", s["width"])
            h = self.norm(x, p + "norm1")
            x = x + getattr(self, "kukulorn_" + layer["type"])(h, p + "mix.", layer["mixer"]) + self.gated(h, p + "mlp.", s["ff"], torch.relu)
        logits = self.norm(x[rows], "final.norm") @ table.T
        return 30.0 * torch.tanh(logits / 30.0)

    def biased(self, h, name, n):
        return self.product(h, name, n) + self.w(name + ".b", n)

    def kukulorn_attention(self, h, p, c):
        d, heads, kv = c["dim"], c["heads"], c["kv_heads"]
        q, k, v = (causal_conv(self.biased(h, p + name, n * d), self.w(f"{p}{name}.conv", n * d, 4)).unflatten(-1, (n, d)) for name, n in (("q", heads), ("k", kv), ("v", kv)))
        freqs = []
        for i in range(d // 2):
            f = 5e5 ** (-2.0 * i / d)
            share = min(1.0, max(0.0, (8192 * f / (2.0 * math.pi) - 1.0) / 3.0))  # whole turns within the original length, from 1 to 4
            freqs.append(share * f + (1.0 - share) * f / 8.0)
        y = attend(over_rms(rotate(q, freqs), self.eps), over_rms(rotate(k, freqs), self.eps), v, c["scale"], cap=c["softcap"]).flatten(2)
        return self.product(y * torch.sigmoid(self.product(h, p + "g", heads * d)), p + "o", self.s["width"])

    def kukulorn_parallel(self, h, p, c):
        left = self.norm(self.kept_window(h, p + "left.", c["left"]), p + "left.out")
        return 0.5 * (left + self.norm(self.state_space(h, p + "right.", c["right"]), p + "right.out"))

    def kept_window(self, h, p, c):
        d, heads, kv = c["dim"], c["heads"], c["kv_heads"]
        q = self.norm(self.biased(h, p + "q", heads * d), p + "q.norm").unflatten(-1, (heads, d))
        k = self.norm(self.biased(h, p + "k", kv * d), p + "k.norm").unflatten(-1, (kv, d))
        v = self.biased(h, p + "v", kv * d).unflatten(-1, (kv, d))
        near, buckets = c["buckets"] // 2, c["buckets"]
        bucket = [n if n < near else min(buckets - 1, near + math.floor(math.log(n / near) / math.log(c["bias_max"] / near) * (buckets - near))) for n in range(h.shape[1])]
        bias = self.w(p + "rel", buckets, heads)[torch.tensor(bucket, device=h.device)].T.contiguous()
        y = attend(q, k, v, c["scale"], window=c["mask"]["size"], keep=c["mask"]["keep_first"], bias=bias)
        y = y * torch.sigmoid(self.product(h, p + "g", heads))[..., None]
        return self.product(y.flatten(2), p + "o", self.s["width"]) + self.w(p + "o.b", self.s["width"])

    def state_space(self, h, p, c):
        heads, vdim, size, groups = c["heads"], c["vdim"], c["state"], c["groups"]
        inner, gn = heads * vdim, groups * size
        z, xbc, step = torch.split(self.product(h, p + "in", 2 * inner + 2 * gn + heads), [inner, inner + 2 * gn, heads], dim=-1)
        xbc = silu(causal_conv(xbc, self.w(p + "conv", inner + 2 * gn, 4)) + self.w(p + "conv.b", inner + 2 * gn))
        x, b, read = torch.split(xbc, [inner, gn, gn], dim=-1)
        x = x.unflatten(-1, (heads, vdim))
        b, read = (y.unflatten(-1, (groups, size)).repeat_interleave(heads // groups, dim=2) for y in (b, read))
        step = torch.nn.functional.softplus(step + self.w(p + "dt_bias", heads), threshold=50.0)
        decay, into = torch.exp(-torch.exp(self.w(p + "A_log", heads)) * step), b * step[..., None]
        state, out = h.new_zeros(h.shape[0], heads, size, vdim), torch.zeros_like(x)
        for t in range(h.shape[1]):
            state = state * decay[:, t, :, None, None] + into[:, t, :, :, None] * x[:, t, :, None, :]
            out[:, t] = torch.matmul(read[:, t, :, None, :], state)[:, :, 0]
        out = (out + self.w(p + "D", heads)[:, None] * x).flatten(2) * silu(z)
        out = over_rms(out.unflatten(-1, (c["norm_groups"], -1)), self.eps).flatten(-2) * self.w(p + "norm", inner)
        return self.product(out, p + "o", self.s["width"])


@torch.no_grad()
def exact(case, seed):
    if "rows" in case:
        return None  # whole numbers
    ids = token_ids(case, seed)
    longest = max(len(row) for row in ids)
    padded = torch.zeros((len(ids), longest), dtype=torch.long)
    for b, row in enumerate(ids):
        padded[b, :len(row)] = torch.tensor(row)
    model = Plain(case)
    # about what a card works in twenty seconds: products in 64 bits, and one token after the other through a recurrence
    products = 2.0 * padded.numel() * sum(n + top * expert for n, _, _, top, expert, *_ in _layers(case))
    if products > 4e14 or (SIZES[case["model"]]["design"] not in ("qwen2", "tiverax") and (longest > 4500 or padded.numel() > 40000)):
        return None
    return {"logits": model.logits(padded.to(DEVICE), [len(row) - 1 for row in ids])}
