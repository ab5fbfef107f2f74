"""What is measured of this engine's speed: rounds of its step function, as a serving program makes them.

A case is one round: ``decoding`` live requests take one token each behind ``context`` tokens (``ragged``: behind
between half of that and all of it) while ``prompts`` new requests of ``prompt`` tokens are taken in, in portions of at
most ``portion`` tokens; then a token is drawn for every row of logits.  ``run`` is such a round through the public
entry points: ``Engine.add_request`` / ``step`` / ``finish`` with ``Lane``s whose tokens lie on the device (what a
scheduler does that queues a round before it has read the tokens of the round before), and ``Sampler.sample_async``.
The tokens that requests decode are drawn beforehand from the seed, so that every implementation computes the same
sequences; the logits are the outcome.  ``score`` asks for the logits of every place of a prompt and draws nothing.

The models have random weights in the sizes of this repository's benchmark: the Falcon-H1 0.5B shape whole, and twelve
layers of the Falcon-H1 7B shape, of the Lutosun (latent attention, experts) and of the Mukutar shape (windowed
attention, delta rule, retention).  A model is loaded once a process and serves every case on it, as in a server.

Drawn tokens are returned by the float32 cases alone: between 16-bit implementations two close logits may change
places, which says nothing about either.
"""
import math

import torch

from macllm_infer_amd import GREEDY, Engine, Lane, Sampler, SamplingParams
from macllm_infer_amd.config import config_from_dict
from macllm_infer_amd.sampling.sampler import SamplerRow
from macllm_infer_amd.weights.random_init import random_tensors

DEVICE = "cuda:0"
PAGE_TOKENS = 16
MAX_CONTEXT = 8192
DECODED = 1500                 # tokens a request decodes before another takes its place
PORTION = 2048                 # prompt tokens a scheduler takes in a round


def _falcon(layers, **sizes):
    # (with multipliers, as the family's configurations have them, by which branches join the stream scaled down)
    raw = dict(
        embedding_multiplier=8.0, ssm_out_multiplier=0.25, mlp_multipliers=[1.0, 0.25],
        architectures=["FalconH1ForCausalLM"], model_type="falcon_h1", hidden_size=1024, num_hidden_layers=layers,
        num_attention_heads=8, num_key_value_heads=2, head_dim=64, intermediate_size=2048, vocab_size=32784,
        max_position_embeddings=MAX_CONTEXT, rms_norm_eps=1e-5, rope_theta=1e11, mamba_n_heads=24, mamba_d_head=64,
        mamba_d_ssm=1536, mamba_d_state=128, mamba_n_groups=1, mamba_d_conv=4, mamba_chunk_size=128,
        mamba_conv_bias=True, mamba_proj_bias=False, mamba_rms_norm=False, attention_bias=False, mlp_bias=False,
        tie_word_embeddings=True)
    return dict(raw, **sizes)


def _lutosun(layers):
    """Sixteen experts a quarter as wide as the Falcon-H1 0.5B shape's feed-forward, three a token beside a shared one."""
    mixer = {"heads": 8, "dim": 64, "rot_dim": 32, "vdim": 64, "q_rank": 512, "kv_rank": 128,
             "rot": {"base": 5e5, "dims": 32}, "scale": 96 ** -0.5}
    mlp = {"kind": "moe", "expert": {"ff": 512, "limit": 7.0}, "router": {"experts": 16, "top": 3, "scale": 1.0},
           "shared": {"ff": 512, "limit": 7.0}}
    # (the embedding enters the stream at order one, times the root of the width, and branches join it scaled down)
    return {"architecture": "Lutosun", "width": 1024, "vocab": 32784, "norm": {"eps": 1e-5}, "residual_mult": 0.25,
            "max_context": MAX_CONTEXT, "logit_softcap": 30.0,
            "embedding": {"scale": 32.0, "bigram": {"buckets": 16384, "mul_prev": 7919, "mul_cur": 104729}},
            "layers": [{"type": "latent_attention", "mixer": mixer, "mlp": mlp} for _ in range(layers)]}


def _mukutar(layers):
    attention = {"type": "attention", "mixer": {"heads": 8, "kv_heads": 2, "dim": 64, "vdim": 64, "scale": 0.125,
                                                "mask": {"size": 1024}}}
    delta = {"type": "general_delta", "mixer": {"heads": 16, "dim": 64, "decay_rank": 64}}
    retention = {"type": "retention", "mixer": {
        "heads": 8, "dim": 64, "vdim": 128, "rot": {"base": 1e6, "dims": 64},
        "decay": [1.0 - 2.0 ** (-5.0 - 4.0 * head / 7.0) for head in range(8)]}}
    kinds = (attention, delta, retention)
    return {"architecture": "Mukutar", "width": 1024, "vocab": 32784, "norm": {"eps": 1e-5}, "max_context": MAX_CONTEXT,
            "layers": [dict(kinds[index % 3], mlp={"kind": "dense", "ff": 2048}) for index in range(layers)]}


# model -> (configuration, dtype, the most requests alive, the most tokens cached)
MODELS = {
    "falcon_0.5b": (_falcon(36), "bfloat16", 272, 1_300_000),
    "falcon_0.5b_f32": (_falcon(36), "float32", 48, 120_000),
    "falcon_7b": (_falcon(12, hidden_size=3072, num_attention_heads=12, head_dim=128, intermediate_size=12288,
                          vocab_size=130049, mamba_n_heads=24, mamba_d_head=128, mamba_d_ssm=3072, mamba_d_state=256,
                          tie_word_embeddings=False), "bfloat16", 80, 400_000),
    "lutosun_0.5b": (_lutosun(12), "bfloat16", 144, 520_000),
    "mukutar_0.5b": (_mukutar(12), "bfloat16", 144, 520_000),
}


def _case(name, model, decoding=0, context=0, ragged=False, prompts=0, prompt=0, portion=PORTION, sampling="greedy",
          score=False):
    return {"name": name, "model": model, "decoding": decoding, "context": context, "ragged": ragged,
            "prompts": prompts, "prompt": prompt, "portion": portion, "sampling": sampling, "score": score}


def listed():
    return [
        # one chat session: the latency of a token
        _case("decode_1", "falcon_0.5b", decoding=1, context=2048),
        # the headline: eight sessions at 2,048-token contexts
        _case("decode_8", "falcon_0.5b", decoding=8, context=2048),
        # a busy server with the default sampling (top-k, top-p, repetition penalty), contexts of all lengths
        _case("decode_64_sampled", "falcon_0.5b", decoding=64, context=2048, ragged=True, sampling="default"),
        # a short question to an idle server: the time to its first token
        _case("prompt_37", "falcon_0.5b", prompts=1, prompt=37),
        # the headline's prompt
        _case("prompt_2048", "falcon_0.5b", prompts=1, prompt=2048),
        # a round of a server that takes in a prompt beside the sessions it serves
        _case("prompt_515_beside_24", "falcon_0.5b", decoding=24, context=1000, ragged=True, prompts=1, prompt=515),
        # logits of every place of a text in float32: evaluation, and the reference that 16-bit results are held against
        _case("score_512_f32", "falcon_0.5b_f32", prompts=1, prompt=512, score=True),
        # a larger model: eight sessions at long contexts
        _case("7b_decode_8", "falcon_7b", decoding=8, context=4096),
        # a long document in two portions
        _case("7b_prompt_4096", "falcon_7b", prompts=1, prompt=4096),
        # a mixture of experts over a latent cache: a batch of an odd size, and two prompts of an odd length in one step
        _case("experts_decode_12", "lutosun_0.5b", decoding=12, context=1500, ragged=True, sampling="default"),
        _case("experts_prompt_2x777", "lutosun_0.5b", prompts=2, prompt=777),
        # linear-state mixers and windowed attention: one prompt of an odd length
        _case("linear_prompt_1999", "mukutar_0.5b", prompts=1, prompt=1999),
    ]


def _log(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


# model -> (most decoding, longest context, longest prompt)
RANGES = {"falcon_0.5b": (64, 4096, 4096), "falcon_0.5b_f32": (8, 1024, 512), "falcon_7b": (16, 4096, 4096),
          "lutosun_0.5b": (32, 2048, 2048), "mukutar_0.5b": (32, 2048, 2048)}


def draw(rng):
    """A round of any of the models: sizes over their ranges, by their logarithm."""
    model = rng.choice(["falcon_0.5b"] * 4 + ["falcon_7b"] * 2 + ["lutosun_0.5b"] * 2 + ["mukutar_0.5b"] * 2
                       + ["falcon_0.5b_f32"])
    most, longest, prompt = RANGES[model]
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "both", "score"])
    case = _case("", model, sampling=rng.choice(["greedy", "default"]) if model != "falcon_0.5b_f32" else "greedy")
    del case["name"]
    if kind in ("decode", "both"):
        case.update(decoding=_log(rng, 1, most), context=_log(rng, 64, longest), ragged=rng.random() < 0.5)
    if kind == "prompt":
        case.update(prompts=rng.choice([1, 1, 1, 2, 3]), portion=rng.choice([PORTION, PORTION, 512]))
        case.update(prompt=_log(rng, 5, min(prompt // case["prompts"], 4 * case["portion"])))
    if kind == "both":
        case.update(prompts=rng.choice([1, 1, 2]), portion=rng.choice([PORTION, PORTION, 256]))
        case.update(prompt=_log(rng, 5, 512))
    if kind == "score":
        case.update(score=True, sampling="greedy", prompts=1, prompt=_log(rng, 16, 512))
    return case


# ------------------------------------------------------------------ the program around the engine

class _Server:
    """A loaded model, its sampler and the names it gives to requests."""

    def __init__(self, model):
        raw, dtype, slots, capacity = MODELS[model]
        config = config_from_dict(raw)
        self.engine = Engine(config=config, tensors=_weights(model), dtype=dtype, kv_cache_block_tokens=PAGE_TOKENS,
                             kv_cache_capacity_tokens=capacity, max_active_sequences=slots)
        self.sampler = Sampler(self.engine.vocab_size, self.engine.device)
        self.pending = None                          # the tokens of the round before, on their way to the host
        self.names = 0

    def name(self):
        self.names += 1
        return f"request-{self.names}"


def _weights(model):
    """The model's weights, the same in every process."""
    raw, dtype, _, _ = MODELS[model]
    return random_tensors(config_from_dict(raw), 0, torch.bfloat16 if dtype == "bfloat16" else torch.float32, "baseline",
                          device=DEVICE)


_servers = {}


def _server(model):
    if model not in _servers:
        _servers[model] = _Server(model)
    return _servers[model]


def _contexts(case):
    """The context length of every decoding request."""
    most, count = case["context"], case["decoding"]
    return [most - (most // 2 * lane // count if case["ragged"] else 0) for lane in range(count)]


def _tokens(case, seed):
    """(each decoding request's context, [DECODED, requests] tokens they go on with, each new prompt)."""
    vocab = MODELS[case["model"]][0].get("vocab_size") or MODELS[case["model"]][0]["vocab"]
    generator = torch.Generator().manual_seed(seed)
    some = lambda *shape: torch.randint(0, vocab, shape, generator=generator, dtype=torch.int32)
    contexts = [some(length).tolist() for length in _contexts(case)]
    follow = some(DECODED, max(case["decoding"], 1))
    return contexts, follow, [some(case["prompt"]).tolist() for _ in range(case["prompts"])]


class _State:
    """Live requests with their contexts in the cache, and the prompts that come in beside them."""

    def __init__(self, case, seed):
        self.case = case
        self.server = _server(case["model"])
        self.contexts, follow, self.prompts = _tokens(case, seed)
        self.follow = follow.to(DEVICE)
        self.params = GREEDY if case["sampling"] == "greedy" else SamplingParams(seed=seed % 1000)
        self.live, self.generated, self.at = [], [], 0
        self.fill()

    def fill(self):
        """New requests behind their contexts."""
        self.release()
        engine = self.server.engine
        self.live = [self.server.name() for _ in self.contexts]
        self.generated = [[] for _ in self.contexts]
        self.at = 0
        for name, tokens in zip(self.live, self.contexts):
            engine.add_request(name)
            for first in range(0, len(tokens), PORTION):
                engine.step([Lane(name, tokens[first:first + PORTION])])

    def release(self):
        for name in self.live:
            self.server.engine.finish(name)
        self.live = []

    def __del__(self):
        self.release()


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    case, server = state.case, state.server
    engine, sampler = server.engine, server.sampler
    incoming = [server.name() for _ in state.prompts]
    for name in incoming:
        engine.add_request(name)
    rounds = []
    for first in range(0, max(case["prompt"], 1), case["portion"]):
        if state.live and state.at == DECODED:       # every request has come to its end: others in their place
            state.fill()
        fed = state.follow[state.at] if state.live else None
        lanes = [Lane(name, [0], [0], feed=(fed, row)) for row, name in enumerate(state.live)]
        rows = [SamplerRow(state.params, context, generated, (fed, row))
                for row, (context, generated) in enumerate(zip(state.contexts, state.generated))]
        for name, prompt in zip(incoming, state.prompts):
            tokens = prompt[first:first + case["portion"]]
            ends = first + len(tokens) == len(prompt)
            if case["score"]:
                want = range(len(tokens))
            else:
                want = [len(tokens) - 1] if ends else []
                rows += [SamplerRow(state.params, prompt, [])] if ends else []
            lanes.append(Lane(name, tokens, want))
        logits = engine.step(lanes)
        state.at += 1 if state.live else 0
        if not logits.shape[0]:                      # a portion that ends no prompt
            continue
        out = {"logits": logits}
        if not case["score"] and rows:
            # (the sampler works in place where it divides by a temperature or counts penalties)
            drawn = sampler.sample_async(logits if state.params is GREEDY else logits.clone(), rows)
            if server.pending is not None:
                server.pending.wait()                # the round before, while the GPU works on this one
            server.pending = drawn
            if case["model"].endswith("f32"):
                out["tokens"] = drawn.device
        rounds.append(out)
    for name in incoming:
        engine.finish(name)
    return rounds


# ------------------------------------------------------------------ what a round cannot do without

def _sizes(model):
    """Per token: matrix elements multiplied outside attention, scans and the head; per round: matrix elements read
    whatever the tokens; one expert's elements; elements cached a token; state elements (float32) of a request;
    multiply-adds of the scan a token; of attention a key seen; the head's elements; the longest window."""
    raw = MODELS[model][0]
    if raw.get("model_type") == "falcon_h1":
        d, q = raw["hidden_size"], raw["num_attention_heads"] * raw["head_dim"]
        kv, inner = raw["num_key_value_heads"] * raw["head_dim"], raw["mamba_d_ssm"]
        n, layers = raw["mamba_d_state"], raw["num_hidden_layers"]
        every = d * (q + 2 * kv) + q * d + d * (2 * inner + 2 * n + raw["mamba_n_heads"]) + inner * d \
            + 3 * d * raw["intermediate_size"]
        return dict(active=layers * every, read=layers * every, expert=0, experts=0, top=0, moe=0,
                    cached=layers * 2 * kv, state=layers * inner * n, scan=layers * 3 * inner * n, seen=layers * 2 * q,
                    head=d * raw["vocab_size"], window=None)
    d, layers = raw["width"], raw["layers"]
    total = dict(active=0, read=0, expert=0, experts=0, top=0, moe=0, cached=0, state=0, scan=0, seen=0,
                 head=d * raw["vocab"], window=None)
    for layer in layers:
        m, mlp = layer["mixer"], layer["mlp"]
        h = m["heads"]
        if layer["type"] == "latent_attention":
            every = d * (m["q_rank"] + m["kv_rank"] + m["rot_dim"]) + m["q_rank"] * h * (m["dim"] + m["rot_dim"]) \
                + h * m["kv_rank"] * (m["dim"] + m["vdim"]) + h * m["vdim"] * d
            total["cached"] += m["kv_rank"] + m["rot_dim"]
            total["seen"] += h * (2 * m["kv_rank"] + m["rot_dim"])
        elif layer["type"] == "attention":
            every = d * m["dim"] * (2 * h + 2 * m["kv_heads"])
            total["cached"] += 2 * m["kv_heads"] * m["dim"]
            total["seen"] += 2 * h * m["dim"]
            total["window"] = m["mask"]["size"]
        elif layer["type"] == "general_delta":
            every = d * 6 * h * m["dim"] + m["decay_rank"] * (d + h * m["dim"])
            total["state"] += h * m["dim"] ** 2
            total["scan"] += 5 * h * m["dim"] ** 2
        else:
            every = d * h * (2 * m["dim"] + 3 * m["vdim"])
            total["state"] += h * m["dim"] * m["vdim"]
            total["scan"] += 2 * h * m["dim"] * m["vdim"]
        if mlp["kind"] == "dense":
            every += 2 * d * mlp["ff"]
        else:
            every += d * (mlp["router"]["experts"] + 1) + 3 * d * mlp["shared"]["ff"]
            total.update(expert=3 * d * mlp["expert"]["ff"], experts=mlp["router"]["experts"], top=mlp["router"]["top"],
                         moe=total["moe"] + 1)
            total["active"] += mlp["router"]["top"] * 3 * d * mlp["expert"]["ff"]
        total["active"] += every
        total["read"] += every
    return total


def _keys(first, tokens, window):
    """Keys that the queries at ``first`` .. ``first + tokens - 1`` see."""
    if window is None:
        return tokens * first + tokens * (tokens + 1) // 2
    return sum(min(position + 1, window) for position in range(first, first + tokens))


def work(case):
    s = _sizes(case["model"])
    element = 4 if case["model"].endswith("f32") else 2
    bytes_, flops = 0, 0
    for first in range(0, max(case["prompt"], 1), case["portion"]):
        taken = min(case["portion"], case["prompt"] - first) if case["prompts"] else 0
        tokens = case["decoding"] + case["prompts"] * taken
        ends = first + taken == case["prompt"]
        rows = case["decoding"] + case["prompts"] * (taken if case["score"] else int(ends and taken > 0))
        # an expert that no token chose is not read: at random, as many are as differ among the choices
        used = s["experts"] * (1.0 - (1.0 - s["top"] / s["experts"]) ** tokens) if s["experts"] else 0.0
        weights = s["read"] + s["moe"] * used * s["expert"] + (s["head"] if rows else 0)
        before = [(length, 1) for length in _contexts(case)] + [(first, taken)] * case["prompts"]
        window = s["window"]
        held = sum(min(length, window) if window else length for length, _ in before)
        keys = sum(_keys(length, count, window) for length, count in before)
        requests = case["decoding"] + case["prompts"]
        fresh = case["prompts"] if first == 0 else 0                 # a new request's state is not read
        bytes_ += element * (weights + s["cached"] * (held + tokens)) + 4 * s["state"] * (2 * requests - fresh) \
            + 4 * rows * (s["head"] // _width(case["model"]))
        flops += 2 * tokens * (s["active"] + s["scan"]) + 2 * s["seen"] * keys + 2 * rows * s["head"]
    return {"bytes": int(bytes_), "flops": int(flops)}


def _width(model):
    return MODELS[model][0].get("hidden_size") or MODELS[model][0]["width"]


def tolerance(case):
    return TOLERANCE[case["model"]]


# Measured, the same sequences taken in whole, in portions and token by token, which sums in other orders and rounds in
# other places: 0.004 and 0.008 on the Falcon-H1 shapes, 0.0015 and 0.009 on the other two, the same bits in float32
# (6.5e-7 off 64 bits).  A choice of experts that rounding turns is a row of logits off by about a hundredth.
TOLERANCE = {"falcon_0.5b": {"rel": 0.016}, "falcon_0.5b_f32": {"rel": 1e-5, "differ": 0.0}, "falcon_7b": {"rel": 0.03},
             "lutosun_0.5b": {"rel": 0.012}, "mukutar_0.5b": {"rel": 0.03}}


# ------------------------------------------------------------------ the same in 64 bits, written out plainly

F = torch.float64


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, base, interleaved=False):
    """x [B, T, ..., D] turned by its place: dimension i with i + D/2, or 2i with 2i + 1."""
    dims, tokens = x.shape[-1], x.shape[1]
    frequency = torch.tensor([1.0 / base ** (i / dims) for i in range(0, dims, 2)], dtype=F).to(torch.float32).to(x)
    angle = torch.arange(tokens, device=x.device).to(F)[:, None] * frequency
    angle = angle.reshape(1, tokens, *([1] * (x.dim() - 3)), dims // 2)
    cos, sin = angle.cos(), angle.sin()
    first, second = (x[..., 0::2], x[..., 1::2]) if interleaved else (x[..., :dims // 2], x[..., dims // 2:])
    turned = first * cos - second * sin, second * cos + first * sin
    return torch.stack(turned, -1).flatten(-2) if interleaved else torch.cat(turned, -1)


def _attend(q, k, v, scale, bias=None, sink=None):
    """q [B, T, H, D], k [B, T, G, D], v [B, T, G, V] -> [B, T, H, V]; bias [H, T, T] holds -inf where masked."""
    tokens, heads, groups = q.shape[1], q.shape[2], k.shape[2]
    out = []
    for q1, k1, v1 in zip(q, k, v):
        spread = lambda x: x.transpose(0, 1).repeat_interleave(heads // groups, 0)
        scores = q1.transpose(0, 1) @ spread(k1).transpose(1, 2).contiguous() * scale
        if bias is None:
            later = torch.ones(tokens, tokens, dtype=torch.bool, device=q.device).triu(1)
            scores = scores.masked_fill(later, -math.inf)
        else:
            scores = scores + bias
        if sink is not None:
            scores = torch.cat([scores, sink.reshape(-1, 1, 1).expand(-1, tokens, 1)], -1)
        out.append((scores.softmax(-1)[..., :tokens] @ spread(v1)).transpose(0, 1))
    return torch.stack(out)


def _scan(x, dt, a, b, c, size=128):
    """S <- exp(dt a) S + dt x b^T, y = S c, in chunks: x [B, T, H, P], dt [B, T, H], a [H], b and c [B, T, N]."""
    batch, tokens, heads, dim = x.shape
    pad = -tokens % size
    x, dt, b, c = (torch.nn.functional.pad(value, (0, 0) * (value.dim() - 2) + (0, pad)) for value in (x, dt, b, c))
    count = (tokens + pad) // size
    xs = (x * dt[..., None]).reshape(batch, count, size, heads, dim).permute(0, 1, 3, 2, 4)      # [B, C, H, Q, P]
    run = (dt * a).reshape(batch, count, size, heads).cumsum(2).permute(0, 1, 3, 2)              # [B, C, H, Q]
    b, c = b.reshape(batch, count, 1, size, -1), c.reshape(batch, count, 1, size, -1)
    later = torch.ones(size, size, dtype=torch.bool, device=x.device).triu(1)
    decay = (run[..., :, None] - run[..., None, :]).masked_fill(later, -math.inf).exp()
    y = (c @ b.transpose(-1, -2) * decay) @ xs
    added = (xs * (run[..., -1:] - run).exp()[..., None]).transpose(-1, -2) @ b                  # [B, C, H, P, N]
    state = torch.zeros_like(added[:, 0])
    for chunk in range(count):
        y[:, chunk] += (c[:, chunk] @ state.transpose(-1, -2)) * run[:, chunk].exp()[..., None]
        state = state * run[:, chunk, :, -1].exp()[..., None, None] + added[:, chunk]
    return y.permute(0, 1, 3, 2, 4).reshape(batch, tokens + pad, heads, dim)[:, :tokens]


def _falcon_rows(raw, get, ids):
    eps, tokens = raw["rms_norm_eps"], ids.shape[1]
    h = get("model.embed_tokens.weight")[ids] * raw["embedding_multiplier"]
    heads, groups, dim = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"]
    inner, state = raw["mamba_d_ssm"], raw["mamba_d_state"]
    for index in range(raw["num_hidden_layers"]):
        at = lambda name: get(f"model.layers.{index}.{name}")
        n = _rms(h, eps) * at("attn_norm.weight")
        project = lambda name, count: (n @ at(f"self_attn.{name}.weight").T).unflatten(-1, (count, dim))
        q, k = _turn(project("q_proj", heads), raw["rope_theta"]), _turn(project("k_proj", groups), raw["rope_theta"])
        attended = _attend(q, k, project("v_proj", groups), dim ** -0.5).flatten(-2) @ at("self_attn.o_proj.weight").T
        z, mixed, dt = (n @ at("mamba.in_proj.weight").T).split([inner, inner + 2 * state, raw["mamba_n_heads"]], -1)
        taps = at("mamba.conv1d.weight").reshape(inner + 2 * state, -1)
        padded = torch.nn.functional.pad(mixed, (0, 0, taps.shape[1] - 1, 0))
        mixed = sum(padded[:, tap:tap + tokens] * taps[:, tap] for tap in range(taps.shape[1])) + at("mamba.conv1d.bias")
        x, b, c = torch.nn.functional.silu(mixed).split([inner, state, state], -1)
        x = x.unflatten(-1, (raw["mamba_n_heads"], -1))
        dt = torch.nn.functional.softplus(dt + at("mamba.dt_bias"), threshold=100.0)
        y = _scan(x, dt, -at("mamba.A_log").reshape(-1).exp(), b, c) + x * at("mamba.D").reshape(-1, 1)
        y = y.flatten(-2) * torch.nn.functional.silu(z)
        h = h + attended + y @ at("mamba.out_proj.weight").T * raw["ssm_out_multiplier"]
        n = _rms(h, eps) * at("ffn_norm.weight")
        gate = torch.nn.functional.silu(n @ at("mlp.gate_proj.weight").T * raw["mlp_multipliers"][0])
        h = h + (gate * (n @ at("mlp.up_proj.weight").T)) @ at("mlp.down_proj.weight").T * raw["mlp_multipliers"][1]
    head = "model.embed_tokens.weight" if raw["tie_word_embeddings"] else "lm_head.weight"
    return _rms(h, eps) * get("model.norm.weight"), get(head), None


def _layer_norm(x, get, name, eps):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], get(name + ".weight"), get(name + ".bias"), eps)


def _lutosun_rows(raw, get, ids):
    eps, hashed = raw["norm"]["eps"], raw["embedding"]["bigram"]
    rows = (ids[:, :-1].long() * hashed["mul_prev"] + ids[:, 1:].long() * hashed["mul_cur"]) % hashed["buckets"]
    rows = torch.cat([torch.full_like(rows[:, :1] if rows.shape[1] else ids[:, :1].long(), hashed["buckets"]), rows], 1)
    h = get("embed.weight")[ids] * raw["embedding"]["scale"] + get("bigram.weight")[rows]
    for index, layer in enumerate(raw["layers"]):
        at = lambda name: get(f"l{index}.{name}")
        m, mlp = layer["mixer"], layer["mlp"]
        heads, dim, rank = m["heads"], m["dim"], m["kv_rank"]
        n = _layer_norm(h, get, f"l{index}.norm1", eps)
        q = (_rms(n @ at("mix.dq.weight").T, eps) * at("mix.dq.norm.weight")) @ at("mix.uq.weight").T
        q = q.unflatten(-1, (heads, -1))
        down = n @ at("mix.dkv.weight").T
        latent = _rms(down[..., :rank], eps) * at("mix.dkv.norm.weight")
        turned = _turn(down[..., None, rank:], m["rot"]["base"], True).expand(-1, -1, heads, -1)
        k = torch.cat([(latent @ at("mix.uk.weight").T).unflatten(-1, (heads, dim)), turned], -1)
        q = torch.cat([q[..., :dim], _turn(q[..., dim:], m["rot"]["base"], True)], -1)
        v = (latent @ at("mix.uv.weight").T).unflatten(-1, (heads, -1))
        h = h + raw["residual_mult"] * (_attend(q, k, v, m["scale"]).flatten(-2) @ at("mix.o.weight").T)
        n = _layer_norm(h, get, f"l{index}.norm2", eps).flatten(0, 1)

        def expert(x, name):
            gate = (x @ at(f"mlp.{name}.gate.weight").T).clamp(max=mlp["expert"]["limit"])
            up = (x @ at(f"mlp.{name}.up.weight").T).clamp(-mlp["expert"]["limit"], mlp["expert"]["limit"])
            return (gate * torch.sigmoid(1.702 * gate) * (up + 1.0)) @ at(f"mlp.{name}.down.weight").T

        scores = (n @ at("mlp.router.weight").T).softmax(-1)
        chosen = (scores + at("mlp.correction")).topk(mlp["router"]["top"], -1).indices
        picked = scores.gather(1, chosen)
        picked = picked / picked.sum(-1, keepdim=True) * mlp["router"]["scale"]
        out = torch.sigmoid(n @ at("mlp.shared.sg.weight").T) * expert(n, "shared")
        for number in range(mlp["router"]["experts"]):
            token, place = (chosen == number).nonzero(as_tuple=True)
            out.index_add_(0, token, expert(n[token], f"e{number}") * picked[token, place][:, None])
        h = h + raw["residual_mult"] * out.view_as(h)
    return _layer_norm(h, get, "final.norm", eps), get("head.weight"), raw["logit_softcap"]


def _mukutar_rows(raw, get, ids):
    eps, tokens = raw["norm"]["eps"], ids.shape[1]
    h = get("embed.weight")[ids]
    distance = (torch.arange(tokens)[:, None] - torch.arange(tokens)[None, :]).to(DEVICE, F)
    for index, layer in enumerate(raw["layers"]):
        at = lambda name: get(f"l{index}.{name}")
        m, heads, dim = layer["mixer"], layer["mixer"]["heads"], layer["mixer"]["dim"]
        n = _rms(h, eps) * (1.0 + at("norm1.weight"))
        mix = lambda name: n @ at(f"mix.{name}.weight").T
        if layer["type"] == "attention":
            q, k, v = ((mix(f"{name}_proj") + at(f"mix.{name}_proj.bias")).unflatten(-1, (-1, dim)) for name in "qkv")
            bias = -at("mix.r1").reshape(-1, 1, 1) * torch.log1p(at("mix.r2").reshape(-1, 1, 1) * distance.clamp(min=0))
            bias = bias.masked_fill((distance < 0) | (distance >= m["mask"]["size"]), -math.inf)
            y = _attend(q, k, v, m["scale"], bias, at("mix.sink")).flatten(-2) @ at("mix.o_proj.weight").T
        elif layer["type"] == "general_delta":
            r, k, v = (mix(name).unflatten(-1, (heads, dim)) for name in "rkv")
            low = torch.tanh(mix("w1")) @ at("mix.w2.weight").T + at("mix.w0")
            decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(low)).unflatten(-1, (heads, dim))
            a = torch.sigmoid(mix("a") + at("mix.a.bias")).unflatten(-1, (heads, dim))
            unit = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            state = torch.zeros(*r.shape[:1], heads, dim, dim, dtype=F, device=h.device)
            outs = []
            for t in range(tokens):
                u = unit[:, t]
                state = (decay[:, t, :, :, None] * state - (a[:, t] * u)[..., None] * (u[..., None, :] @ state)
                         + k[:, t, :, :, None] * v[:, t, :, None, :])
                outs.append((r[:, t, :, None, :] @ state).squeeze(-2))
            y = _rms(torch.stack(outs, 1), eps).flatten(-2) * at("mix.norm.weight")
            y = (y * torch.sigmoid(mix("g"))) @ at("mix.o.weight").T
        else:
            q, k = (_turn(mix(name).unflatten(-1, (heads, dim)), m["rot"]["base"]) for name in "qk")
            v = mix("v").unflatten(-1, (heads, -1)).transpose(1, 2)
            rate = torch.tensor(m["decay"], dtype=F, device=h.device).reshape(-1, 1, 1)
            kept = torch.where(distance < 0, 0.0, rate ** distance.clamp(min=0))
            weights = q.transpose(1, 2) @ k.transpose(1, 2).transpose(-1, -2).contiguous() * dim ** -0.5 * kept
            y = _rms((weights @ v).transpose(1, 2), eps).flatten(-2)
            y = (y * torch.nn.functional.silu(mix("g"))) @ at("mix.o.weight").T
        h = h + y * at("ls1")
        n = _rms(h, eps) * (1.0 + at("norm2.weight"))
        z, c = n @ at("mlp.up.weight").T, at("mlp.act")
        z = c[0] * _rms(z, eps) + c[1] * _rms(z * z, eps) + c[2] * _rms(z * z * z, eps) + c[3]
        h = h + (z @ at("mlp.down.weight").T) * at("ls2")
    return _rms(h, eps) * (1.0 + get("final.norm.weight")), get("head.weight"), None


def exact(case, seed):
    raw, weights = MODELS[case["model"]][0], _weights(case["model"])
    get = lambda name: weights[name].to(F)
    rows_of = {"Lutosun": _lutosun_rows, "Mukutar": _mukutar_rows}.get(raw.get("architecture"), _falcon_rows)
    contexts, follow, prompts = _tokens(case, seed)
    steps = -(-max(case["prompt"], 1) // case["portion"])
    # every sequence as it stands at the round's end, and its wanted places step by step
    sequences, wanted = [], []
    for lane, context in enumerate(contexts):
        sequences.append(context + follow[:steps, lane].tolist())
        wanted.append([[len(context) + step] for step in range(steps)])
    for prompt in prompts:
        sequences.append(prompt)
        every = [range(first, min(first + case["portion"], len(prompt))) for first in range(0, len(prompt), case["portion"])]
        wanted.append([list(places) if case["score"] else [len(prompt) - 1] if places[-1] == len(prompt) - 1 else []
                       for places in every])
    found = [[None] * len(sequences) for _ in range(steps)]
    longest = max(len(sequence) for sequence in sequences)
    together = max(1, 16384 // longest)
    for first in range(0, len(sequences), together):
        group = sequences[first:first + together]
        ids = torch.zeros(len(group), longest, dtype=torch.long)      # (what follows a sequence's end changes nothing before it)
        for lane, sequence in enumerate(group):
            ids[lane, :len(sequence)] = torch.tensor(sequence)
        hidden, head, cap = rows_of(raw, get, ids.to(DEVICE))
        for lane in range(len(group)):
            for step in range(steps):
                logits = hidden[lane, wanted[first + lane][step]] @ head.T
                found[step][first + lane] = logits if cap is None else cap * torch.tanh(logits / cap)
        del hidden
    out = []
    for logits in (torch.cat(step) for step in found):
        if not logits.shape[0]:
            continue
        out.append({"logits": logits})
        if case["model"].endswith("f32") and not case["score"]:
            out[-1]["tokens"] = None
    return out
