"""Mixers that carry a matrix-valued state per head from token to token instead of a cache of keys:
retention and lightning attention (a fixed decay per head), gated linear attention (a decay per key channel) and the
generalized delta rule (a decay per key channel and a removal of what the state holds along the unit key).  All keep
their state [heads, value dim, key dim] in float32 in the request's state slot and run through one scan kernel
(``ops.linear_state_scan``), for prompt portions and for single decoded tokens alike, but that retention and the delta
rule take bfloat16 portions to the float32 matrix cores where that pays (``runs_pay``, ``ops.linear_matrix_scan``) and
lightning attention has chunks of its own; rotation, decays, gates of the recurrence and unit keys are formed in float32
inside it.  The head-wise root-mean-square norm, its weight and the output gate are one more launch.
"""
from __future__ import annotations

from typing import Optional

import torch

from ..cache.manager import StateNeed
from ..kernels import ops
from ..kernels.limits import GRID_MOST, LINEAR_STATE_MAX_KEY_DIM, beyond
from ..weights.loader import Expect
from .base import BuildContext, Mixer, part_class, register_part
from .linear import Linear


CHUNK_TOKENS = 128      # lanes longer than this scan in chunks of this many tokens, side by side


def scan_chunks(step):
    """The step's lanes cut into chunks when one of them is long enough for the scan in passes to pay, else None
    (the scan then walks every lane from end to end, which is what steps of single tokens and short portions want)."""
    if step.max_query_len <= CHUNK_TOKENS:
        return None
    return chunk_table(step)


def chunk_table(step):
    """The step's lanes cut into chunks of ``CHUNK_TOKENS`` tokens."""
    table = step.chunk_tables.get(CHUNK_TOKENS)
    if table is not None:
        return table
    key = ("linear_state_chunks", CHUNK_TOKENS)              # a step that was packed without the table
    if key not in step.derived:
        step.derived[key] = ops.SsdChunks(step.lane_lengths, CHUNK_TOKENS, step.token_ids.device)
    return step.derived[key]


# (delta rule, key channels) -> the tokens from which on runs on the matrix cores pay; the lanes x heads up to which they do
# in a step of up to 8 lanes that holds so many tokens a lane; the lanes x heads a token of the average lane, of at most so many tokens,
# up to which they do in any case.  See ``runs_pay``.
RUNS_PAY = {(True, 64): (32, 128, 10, 3.0, 128), (True, 128): (48, 64, 40, 1.0, 256),
            (False, 64): (32, 128, 10, 3.0, 128), (False, 128): (64, 128, 40, 0.9, 256)}


def runs_pay(tokens: int, lanes: int, heads: int, key_dim: int, delta: bool) -> bool:
    """Whether a step of so many tokens in so many lanes (those of a captured step, which does not know how its tokens fall
    into lanes) is faster in runs on the matrix cores than token by token, end to end or in chunks of 128.

    A lane costs a run's matrices however few tokens it has, the walk its longest lane.  us a layer, token by token | in
    runs, steps of a capacity (token by token: end to end up to 128 tokens, in chunks beyond):

    * delta rule, 16 heads of 64: one lane of 32 tokens 33 | 23, 100 96 | 23, 2,048 244 | 104; 3 single tokens beside 60 59 |
      21, beside 512 169 | 46; 8 lanes of 16 18 | 29, of 32 30 | 31, of 64 52 | 37; 16 lanes of 32 31 | 56, of 64 53 | 64,
      of 128 111 | 80; 32 lanes of 8 18 | 97, of 64 69 | 120.  48 heads: 4 lanes of 64 53 | 50, 8 of 64 65 | 90, of 128 123 | 117.
    * delta rule, heads of 128: 8 of them, one lane of 32 36 | 37, of 48 52 | 37, of 2,048 354 | 241; 8 lanes of 64 69 | 56, 16
      of 64 73 | 103, of 128 136 | 127; 3 single tokens beside 256 227 | 59.  32 heads: 2 lanes of 64 68 | 56, 4 of 64 73 |
      103, of 128 136 | 127, 8 of 128 142 | 257, of 256 676 | 467.
    * retention, 8 heads of 64: one lane of 32 22 | 20, 2,048 125 | 48; 8 lanes of 16 13 | 21, of 32 23 | 21; 16 of 32 24 | 28, of
      64 39 | 30; 32 of 64 45 | 46.  16 heads of 128 (values of 256): one lane of 48 37 | 38, of 64 49 | 39; 4 lanes of 64 46 |
      54, of 128 85 | 62; 8 of 64 58 | 65, of 128 97 | 80; 3 single tokens beside 256 139 | 67."""
    least, sure, few, slope, longest = RUNS_PAY[delta, key_dim]
    return tokens >= least and ((lanes <= 8 and lanes * heads <= sure and tokens >= few * lanes)
                                or (lanes * heads <= slope * min(tokens / lanes, longest) and tokens >= least * lanes))


def run_scan(u: torch.Tensor, step, columns: dict, recurrence: dict) -> None:
    """The scan of retention or the delta rule: a run of tokens at a time on the float32 matrix cores for prompt portions in
    bfloat16 whose heads those kernels cover, else token by token (single tokens, many short lanes, float32, other sizes)."""
    floor = recurrence.get("decay_floor")
    lanes, tokens, _ = step.sizes
    heads, sizes = columns["num_heads"], (columns["key_dim"], columns["value_dim"])
    if (u.is_cuda and step.max_query_len > 1 and ops.linear_matrix_supported(u.dtype, *sizes, floor)
            and runs_pay(tokens, lanes, heads, sizes[0], floor is not None)
            and ops.linear_matrix_bytes(tokens, lanes, heads, *sizes, floor is not None) <= ops.LINEAR_MATRIX_MOST_BYTES
            and columns["state"].data_ptr() % 16 == 0):
        ops.linear_matrix_scan(u, **columns, **recurrence, slot_ids=step.slot_ids, chunks=chunk_table(step))
        return
    ops.linear_state_scan(u, **columns, **recurrence, cu_seqlens=step.cu_seqlens, slot_ids=step.slot_ids,
                          max_query_len=step.max_query_len, chunks=scan_chunks(step))


def scan_modules(modules: tuple, key_dim: int, value_dim: int) -> tuple:
    """Without the kernels of runs on the matrix cores for heads that they do not cover."""
    covered = key_dim in ops.LINEAR_MATRIX_KEY_DIMS and value_dim % 16 == 0
    return tuple(name for name in modules if covered or name != "linear_matrix")


@register_part("retention")
class Retention(Mixer):
    """[q | k | v | g] = one projection of the normed rows; q and k rotated by position, k scaled;
    S <- decay[h] S + k v^T, o = S^T q per head; o / rms(o) per head, times SiLU(g), output projection."""
    graph_safe = True
    kernel_modules = ("common", "linear_state", "linear_matrix", "gemm")
    chunk_tokens = CHUNK_TOKENS

    @classmethod
    def modules_of(cls, spec) -> tuple:
        return scan_modules(cls.kernel_modules, spec.key_dim, spec.value_dim)

    @classmethod
    def expected_tensors(cls, spec, prefix: str, hidden_size: int):
        keys, values = spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        return [Expect(f"{prefix}.q.weight", ((keys, hidden_size),)),
                Expect(f"{prefix}.k.weight", ((keys, hidden_size),)),
                Expect(f"{prefix}.v.weight", ((values, hidden_size),)),
                Expect(f"{prefix}.g.weight", ((values, hidden_size),)),
                Expect(f"{prefix}.o.weight", ((hidden_size, values),))]

    @classmethod
    def limits(cls, spec, hidden_size: int):
        return (beyond("retention", "key_dim", spec.key_dim, LINEAR_STATE_MAX_KEY_DIM,
                       "a column of a head's state is spread over at most one wave")
                + beyond("retention", "num_heads", spec.num_heads, GRID_MOST, "heads index a dimension of the launch")
                + part_class(spec.position).limits(spec.position, spec.key_dim))

    @classmethod
    def cache_needs(cls, spec):
        return [StateNeed("state", (spec.num_heads, spec.value_dim, spec.key_dim), "float32")]

    def __init__(self, spec, prefix: str, tensors, build: BuildContext):
        self.spec = spec
        get = lambda name: tensors.get(f"{prefix}.{name}")
        self.in_proj = Linear([get("q.weight"), get("k.weight"), get("v.weight"), get("g.weight")],
                              [None, None, None, None], build)
        self.out_proj = Linear([get("o.weight")], [None], build)
        self.decay = torch.tensor(spec.decay, dtype=torch.float64).to(torch.float32).to(build.device)
        position = part_class(spec.position)(spec.position, spec.key_dim, build)
        rotation = position.fused_rotation()
        if rotation is None:
            raise ValueError(f"retention turns q and k inside its scan: the position encoding {spec.position.kind!r} "
                             "is no rotation by position")
        self.inv_freq, self.rotary_dim = rotation

    def forward(self, x: torch.Tensor, step, cache) -> torch.Tensor:
        spec = self.spec
        keys, values = spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        u = self.in_proj(x)                                              # [T, q | k | v | g]
        raw = torch.empty((x.shape[0], values), dtype=torch.float32, device=x.device)
        run_scan(u, step, dict(q_col=0, k_col=keys, v_col=2 * keys, num_heads=spec.num_heads, key_dim=spec.key_dim,
                               value_dim=spec.value_dim, state=cache.states["state"], out=raw),
                 dict(head_decay=self.decay, key_scale=spec.key_scale, positions=step.positions, inv_freq=self.inv_freq,
                      rotary_dim=self.rotary_dim))
        gated = torch.empty((x.shape[0], values), dtype=u.dtype, device=x.device)
        ops.head_norm_gate(raw, u[:, 2 * keys + values:], None, spec.num_heads, spec.norm_eps, "silu", gated)
        return self.out_proj(gated)


@register_part("general_delta")
class GeneralDelta(Mixer):
    """[r | k | v | g | a | w1] = one projection of the normed rows (a with its bias);
    decay logits = w2 tanh(w1 part) in float32; inside the scan w = exp(-floor * sigmoid(logits + w0)),
    a = sigmoid(a part), u = k / sqrt(sum k^2 + key_eps), S <- diag(w) S - (a u)(u^T S) + k v^T, o = S^T r;
    then o / rms(o) per head times the weight ``norm``, times sigmoid(g), output projection."""
    graph_safe = True
    kernel_modules = ("common", "linear_state", "linear_matrix", "gemm")
    chunk_tokens = CHUNK_TOKENS

    @classmethod
    def modules_of(cls, spec) -> tuple:
        return scan_modules(cls.kernel_modules, spec.head_dim, spec.head_dim)

    @classmethod
    def expected_tensors(cls, spec, prefix: str, hidden_size: int):
        inner = spec.num_heads * spec.head_dim
        rank = -1 if spec.decay_rank is None else spec.decay_rank
        return [Expect(f"{prefix}.r.weight", ((inner, hidden_size),)),
                Expect(f"{prefix}.k.weight", ((inner, hidden_size),)),
                Expect(f"{prefix}.v.weight", ((inner, hidden_size),)),
                Expect(f"{prefix}.g.weight", ((inner, hidden_size),)),
                Expect(f"{prefix}.a.weight", ((inner, hidden_size),)),
                Expect(f"{prefix}.a.bias", ((inner,),), init="bias"),
                Expect(f"{prefix}.w1.weight", ((rank, hidden_size),)),
                Expect(f"{prefix}.w2.weight", ((inner, rank),)),
                Expect(f"{prefix}.w0", ((inner,),), init="logit"),
                Expect(f"{prefix}.norm.weight", ((inner,),), init="norm"),
                Expect(f"{prefix}.o.weight", ((hidden_size, inner),))]

    @classmethod
    def limits(cls, spec, hidden_size: int):
        return (beyond("general_delta", "head_dim", spec.head_dim, LINEAR_STATE_MAX_KEY_DIM,
                       "a column of a head's state is spread over at most one wave")
                + beyond("general_delta", "num_heads", spec.num_heads, GRID_MOST, "heads index a dimension of the launch"))

    @classmethod
    def cache_needs(cls, spec):
        return [StateNeed("state", (spec.num_heads, spec.head_dim, spec.head_dim), "float32")]

    def __init__(self, spec, prefix: str, tensors, build: BuildContext):
        self.spec = spec
        get = lambda name: tensors.get(f"{prefix}.{name}")
        if get("w1.weight").shape[0] != get("w2.weight").shape[1]:
            raise ValueError(f"{prefix}: the decay's two projections do not fit each other: "
                             f"{tuple(get('w1.weight').shape)} and {tuple(get('w2.weight').shape)}")
        self.rank = get("w1.weight").shape[0]
        self.in_proj = Linear([get("r.weight"), get("k.weight"), get("v.weight"), get("g.weight"), get("a.weight"),
                               get("w1.weight")], [None, None, None, None, get("a.bias"), None], build)
        self.decay_proj = Linear([get("w2.weight")], [None], build)
        self.out_proj = Linear([get("o.weight")], [None], build)
        f32 = lambda tensor: tensor.to(torch.float32).contiguous().to(build.device)
        self.decay_bias = f32(get("w0"))
        self.norm_weight = f32(get("norm.weight"))

    def forward(self, x: torch.Tensor, step, cache) -> torch.Tensor:
        spec = self.spec
        inner = spec.num_heads * spec.head_dim
        u = self.in_proj(x)                                              # [T, r | k | v | g | a | w1]
        bent = torch.empty((x.shape[0], self.rank), dtype=u.dtype, device=x.device)
        ops.tanh_rows(u[:, 5 * inner:], bent)
        logits = ops.linear(bent, self.decay_proj.weight, None, keep_float32=True)     # float32 [T, inner]
        raw = torch.empty((x.shape[0], inner), dtype=torch.float32, device=x.device)
        run_scan(u, step, dict(q_col=0, k_col=inner, v_col=2 * inner, num_heads=spec.num_heads, key_dim=spec.head_dim,
                               value_dim=spec.head_dim, state=cache.states["state"], out=raw),
                 dict(removal_col=4 * inner, decay_logits=logits, decay_bias=self.decay_bias, decay_floor=spec.decay_floor,
                      key_eps=spec.key_eps))
        gated = torch.empty((x.shape[0], inner), dtype=u.dtype, device=x.device)
        ops.head_norm_gate(raw, u[:, 3 * inner:4 * inner], self.norm_weight, spec.num_heads, spec.norm_eps, "sigmoid",
                           gated)
        return self.out_proj(gated)


@register_part("gated_linear_attention")
class GatedLinearAttention(Mixer):
    """[q | k | v | g | a1] = one projection of the normed rows; decay logits z = a2 (a1 part) in float32; inside the
    scan q is multiplied by ``query_scale`` and alpha = sigmoid(z + bias)^(1 / temperature) = exp(log sigmoid / temperature)
    decays every key channel of the state on its own, S <- diag(alpha) S + k v^T, o = S^T q; then o / rms(o) per head
    times a weight of value_dim numbers that the heads share, times SiLU(g), output projection."""
    graph_safe = True
    kernel_modules = ("common", "linear_state", "gemm")
    chunk_tokens = CHUNK_TOKENS

    @classmethod
    def expected_tensors(cls, spec, prefix: str, hidden_size: int):
        keys, values = spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        rank = -1 if spec.decay_rank is None else spec.decay_rank
        return [Expect(f"{prefix}.q.weight", ((keys, hidden_size),)),
                Expect(f"{prefix}.k.weight", ((keys, hidden_size),)),
                Expect(f"{prefix}.v.weight", ((values, hidden_size),)),
                Expect(f"{prefix}.g.weight", ((values, hidden_size),)),
                Expect(f"{prefix}.a1.weight", ((rank, hidden_size),)),
                Expect(f"{prefix}.a2.weight", ((keys, rank),)),
                Expect(f"{prefix}.a2.bias", ((keys,),), init="logit"),
                Expect(f"{prefix}.norm.weight", ((spec.value_dim,),), init="norm"),
                Expect(f"{prefix}.o.weight", ((hidden_size, values),))]

    @classmethod
    def limits(cls, spec, hidden_size: int):
        return (beyond("gated_linear_attention", "key_dim", spec.key_dim, LINEAR_STATE_MAX_KEY_DIM,
                       "a column of a head's state is spread over at most one wave")
                + beyond("gated_linear_attention", "num_heads", spec.num_heads, GRID_MOST,
                         "heads index a dimension of the launch"))

    @classmethod
    def cache_needs(cls, spec):
        return [StateNeed("state", (spec.num_heads, spec.value_dim, spec.key_dim), "float32")]

    def __init__(self, spec, prefix: str, tensors, build: BuildContext):
        self.spec = spec
        get = lambda name: tensors.get(f"{prefix}.{name}")
        if get("a1.weight").shape[0] != get("a2.weight").shape[1]:
            raise ValueError(f"{prefix}: the decay's two projections do not fit each other: "
                             f"{tuple(get('a1.weight').shape)} and {tuple(get('a2.weight').shape)}")
        self.rank = get("a1.weight").shape[0]
        self.in_proj = Linear([get("q.weight"), get("k.weight"), get("v.weight"), get("g.weight"), get("a1.weight")],
                              [None, None, None, None, None], build)
        self.decay_proj = Linear([get("a2.weight")], [None], build)
        self.out_proj = Linear([get("o.weight")], [None], build)
        f32 = lambda tensor: tensor.to(torch.float32).contiguous().to(build.device)
        self.decay_bias = f32(get("a2.bias"))
        self.norm_weight = f32(get("norm.weight")).repeat(spec.num_heads).contiguous()      # one copy a head

    def forward(self, x: torch.Tensor, step, cache) -> torch.Tensor:
        spec = self.spec
        keys, values = spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        u = self.in_proj(x)                                              # [T, q | k | v | g | a1]
        inner = u[:, 2 * keys + 2 * values:]
        if inner.stride(0) % 8 != 0 or inner.data_ptr() % 16 != 0:      # the product wants whole 16-byte pieces
            inner = inner.contiguous()
        logits = ops.linear(inner, self.decay_proj.weight, None, keep_float32=True)      # float32 [T, H * dk]
        raw = torch.empty((x.shape[0], values), dtype=torch.float32, device=x.device)
        ops.linear_state_scan(u, q_col=0, k_col=keys, v_col=2 * keys, num_heads=spec.num_heads, key_dim=spec.key_dim,
                              value_dim=spec.value_dim, state=cache.states["state"], cu_seqlens=step.cu_seqlens,
                              slot_ids=step.slot_ids, out=raw, max_query_len=step.max_query_len,
                              decay_logits=logits, decay_bias=self.decay_bias, gate_power=1.0 / spec.decay_temperature,
                              query_scale=spec.query_scale, chunks=scan_chunks(step))
        gated = torch.empty((x.shape[0], values), dtype=u.dtype, device=x.device)
        ops.head_norm_gate(raw, u[:, 2 * keys + values:2 * keys + 2 * values], self.norm_weight, spec.num_heads,
                           spec.norm_eps, "silu", gated)
        return self.out_proj(gated)


@register_part("lightning_attention")
class LightningAttention(Mixer):
    """[q | k | v | g] = one projection of the normed rows; inside the scan q, k and v go through SiLU (float32),
    S <- decay[h] S + k v^T, o = S^T q per head; then all heads' o / rms(o) over their whole width, times one weight, times
    sigmoid(g), output projection.  Prompt portions in bfloat16 are worked on chunk by chunk on the matrix cores where
    the heads' sizes allow; single tokens, short portions, float32 and other sizes walk token by token."""
    graph_safe = True
    takes_tail = True
    kernel_modules = ("common", "linear_state", "linear_chunk", "gemm")
    chunk_tokens = CHUNK_TOKENS
    matrix_from = 32            # tokens of the longest lane from which on the matrix cores are faster than the walk

    @classmethod
    def expected_tensors(cls, spec, prefix: str, hidden_size: int):
        keys, values = spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        return [Expect(f"{prefix}.q.weight", ((keys, hidden_size),)),
                Expect(f"{prefix}.k.weight", ((keys, hidden_size),)),
                Expect(f"{prefix}.v.weight", ((values, hidden_size),)),
                Expect(f"{prefix}.g.weight", ((values, hidden_size),)),
                Expect(f"{prefix}.norm.weight", ((values,),), init="norm"),
                Expect(f"{prefix}.o.weight", ((hidden_size, values),))]

    @classmethod
    def limits(cls, spec, hidden_size: int):
        return (beyond("lightning_attention", "key_dim", spec.key_dim, LINEAR_STATE_MAX_KEY_DIM,
                       "a column of a head's state is spread over at most one wave")
                + beyond("lightning_attention", "num_heads", spec.num_heads, GRID_MOST,
                         "heads index a dimension of the launch"))

    @classmethod
    def cache_needs(cls, spec):
        return [StateNeed("state", (spec.num_heads, spec.value_dim, spec.key_dim), "float32")]

    def __init__(self, spec, prefix: str, tensors, build: BuildContext):
        self.spec = spec
        get = lambda name: tensors[f"{prefix}.{name}"]
        self.in_proj = Linear([get("q.weight"), get("k.weight"), get("v.weight"), get("g.weight")],
                              [None, None, None, None], build)
        self.out_proj = Linear([get("o.weight")], [None], build)
        self.decay = torch.tensor(spec.decay, dtype=torch.float64).to(torch.float32).to(build.device)
        self.norm_weight = get("norm.weight").to(torch.float32).contiguous().to(build.device)

    def forward(self, x: torch.Tensor, step, cache, tail=None) -> Optional[torch.Tensor]:
        spec = self.spec
        keys, values = spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        u = self.in_proj(x)                                              # [T, q | k | v | g]
        raw = torch.empty((x.shape[0], values), dtype=torch.float32, device=x.device)
        columns = dict(q_col=0, k_col=keys, v_col=2 * keys, num_heads=spec.num_heads, key_dim=spec.key_dim,
                       value_dim=spec.value_dim, state=cache.states["state"], slot_ids=step.slot_ids, out=raw,
                       head_decay=self.decay, silu=True)
        if (step.max_query_len >= self.matrix_from and ops.linear_chunk_supported(u.dtype, spec.key_dim, spec.value_dim)
                and u.stride(0) % 8 == 0 and u.data_ptr() % 16 == 0):
            ops.linear_chunk_scan(u, **columns, chunks=chunk_table(step))
        else:
            ops.linear_state_scan(u, **columns, cu_seqlens=step.cu_seqlens, max_query_len=step.max_query_len,
                                  chunks=scan_chunks(step))
        gated = torch.empty((x.shape[0], values), dtype=u.dtype, device=x.device)
        ops.head_norm_gate(raw, u[:, 2 * keys + values:], self.norm_weight, 1, spec.norm_eps, "sigmoid", gated)
        if tail is not None and tail.project(self.out_proj, gated):
            return None
        return self.out_proj(gated)
