"""The work a user of this package has it do, as timed cases through its
public entry points: decode steps of the fused recurrence, prompts through
the chunked update and the short-run scan, the layer's core, the quantized
projections, and two whole-layer calls.

``listed()`` holds the cases, ``draw()`` gives further ones of the same
ranges; ``prepare`` / ``run`` make and run one, ``work`` is what a pass
cannot do without, ``tolerance`` the agreement two correct implementations
reach, and ``exact`` the same outputs in float64 from plain torch.
"""

from __future__ import annotations

import copy
import math
import random

import torch

import mlx_lean_moe_amd as gdn

DEV = "cuda"
CONV_K = 4
CHUNK = 64
EPS = 1e-6
ACT = {"bf16": torch.bfloat16, "f32": torch.float32}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # one sequence's token: the reference's own decode mode (its states
        # are replaced, not updated in place)
        dict(name="decode_1", kind="decode", batch=1, pool=0, value_heads=32, act="bf16", norm=True),
        # a serving step over part of a pool, float32 activations (what the
        # reference's layers carry), sequences at scattered slots
        dict(name="decode_48_of_100_f32", kind="decode", batch=48, pool=100, value_heads=32, act="f32",
             norm=True),
        # the largest decode batch: 1 GB of state
        dict(name="decode_256_hv64", kind="decode", batch=256, pool=256, value_heads=64, act="bf16", norm=True),
        # one long prompt from an empty state
        dict(name="update_4096", kind="update", runs=1, shortest=4096, longest=4096, lens_seed=0, packed=False,
             value_heads=32, dtype="bf16", state=False),
        # a batch of prompts of mixed length packed into one stream, each
        # continuing from a state
        dict(name="update_packed_16", kind="update", runs=16, shortest=128, longest=8192, lens_seed=3,
             packed=True, value_heads=32, dtype="bf16", state=True),
        # three equal prompts of an odd length, float32
        dict(name="update_f32_3x777", kind="update", runs=3, shortest=777, longest=777, lens_seed=0,
             packed=False, value_heads=32, dtype="f32", state=True),
        # a run too short for the chunked path: a short prompt's tail, a
        # draft being verified
        dict(name="scan_41", kind="scan", tokens=41, key_heads=16, value_heads=32, key_dim=128, value_dim=128,
             dtype="bf16"),
        # everything between the projections for one float32 prompt
        dict(name="core_f32_1531", kind="core", runs=1, shortest=1531, longest=1531, lens_seed=0,
             value_heads=32, act="f32"),
        # a projection at a batch above the decode sizes (200 sequences, or a
        # short prompt)
        dict(name="linear_200", kind="linear", rows=200, out=12352, hidden=2048, mode="affine", bits=4,
             group=64, act="bf16"),
        # a prompt's projection with float32 activations
        dict(name="linear_f32_777", kind="linear", rows=777, out=12352, hidden=2048, mode="affine", bits=4,
             group=64, act="f32"),
        # whole layer, one token for 64 active sequences out of 256 slots,
        # replayed from its graph
        dict(name="layer_decode_64", kind="layer_decode", batch=64, pool=256, hidden=2048, act="bf16"),
        # whole layer over one prompt of an odd length
        dict(name="layer_prompt_1999", kind="layer_prompt", tokens=1999, hidden=2048, act="bf16"),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("decode", "update", "update", "scan", "core", "linear", "linear", "layer_decode",
                       "layer_prompt"))
    if kind == "decode":
        batch = _log_int(rng, 1, 256)
        pool = rng.choice((0, batch, batch + _log_int(rng, 1, 256)))
        return dict(kind=kind, batch=batch, pool=pool, value_heads=rng.choice((32, 64) if batch + pool <= 256 else (32,)),
                    act=rng.choice(("bf16", "bf16", "f32")), norm=rng.random() < 0.75)
    if kind in ("update", "core"):
        runs = rng.choice((1, 1, _log_int(rng, 2, 32)))
        longest = _log_int(rng, 64, 8192 if kind == "update" else 4096)
        # at most 48 k tokens in all, less than the largest listed case
        longest = max(64, min(longest, 49152 // runs))
        if runs == 1:
            shortest = longest
        else:
            shortest = rng.choice((longest, max(64, longest // rng.randint(2, 16))))
        case = dict(kind=kind, runs=runs, shortest=shortest, longest=longest, lens_seed=rng.randrange(1000),
                    value_heads=rng.choice((16, 32, 32, 64) if runs * longest <= 16384 else (16, 32)))
        if kind == "update":
            case.update(packed=shortest != longest or rng.random() < 0.3, dtype=rng.choice(("bf16", "bf16", "f32")),
                        state=rng.random() < 0.7)
        else:
            case.update(act=rng.choice(("bf16", "f32")))
        return case
    if kind == "scan":
        key_dim, value_dim = rng.choice(((128, 128), (128, 128), (64, 64), (256, 256), (128, 17)))
        return dict(kind=kind, tokens=_log_int(rng, 2, 63 if key_dim == value_dim == 128 else 512), key_heads=16,
                    value_heads=rng.choice((16, 32)), key_dim=key_dim, value_dim=value_dim,
                    dtype=rng.choice(("bf16", "f32")))
    if kind == "linear":
        mode, bits, group = rng.choice((("affine", 4, 64), ("affine", 4, 64), ("affine", 4, 64), ("affine", 4, 32),
                                        ("affine", 8, 64), ("affine", 6, 64), ("affine", 3, 128), ("mxfp4", 4, 32),
                                        ("mxfp8", 8, 32), ("nvfp4", 4, 16)))
        act = rng.choice(("bf16", "bf16", "f32"))
        hidden = rng.choice((1024, 2048, 2048, 3072, 4096))
        # the stacked input projection of a hidden width, or its out_proj
        out, width = rng.choice(((12352, hidden), (hidden, 4096)))
        return dict(kind=kind, rows=_log_int(rng, 1, 4096 if act == "bf16" else 1024), out=out, hidden=width,
                    mode=mode, bits=bits, group=group, act=act)
    if kind == "layer_decode":
        batch = _log_int(rng, 1, 200)
        return dict(kind=kind, batch=batch, pool=batch + rng.randint(0, 100), hidden=rng.choice((1024, 2048, 4096)),
                    act="bf16")
    return dict(kind=kind, tokens=_log_int(rng, 2, 4096), hidden=rng.choice((1024, 2048, 4096)),
                act=rng.choice(("bf16", "bf16", "f32")))


def _dims(case) -> gdn.LinearAttentionDims:
    return gdn.LinearAttentionDims(16, case.get("value_heads", 32), 128, 128, CONV_K)


def _lens(case) -> list[int]:
    rng = random.Random(case["lens_seed"])
    return [rng.randint(case["shortest"], case["longest"]) for _ in range(case["runs"])]


def _offsets(lens: list[int]) -> list[int]:
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return out


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


class _Rand:
    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.py = random.Random(seed)

    def normal(self, *shape, dtype=torch.float32, scale=1.0):
        return (torch.randn(*shape, generator=self.g, device=DEV) * scale).to(dtype)

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo


def _gate_params(r: _Rand, heads: int) -> dict:
    """Decay rates A in [1, 16) and their time-step biases."""
    return dict(A_log=r.uniform(0.0, math.log(16.0), heads), dt_bias=r.uniform(-1.0, 1.0, heads))


def _layer_params(r: _Rand, dims) -> dict:
    return dict(conv_w=r.normal(dims.conv_dim, CONV_K, scale=0.2).to(torch.bfloat16).float(),
                norm_w=r.uniform(0.5, 1.5, dims.value_head_dim), **_gate_params(r, dims.num_value_heads))


def _unit(t: torch.Tensor, scale: float = 1.0) -> torch.Tensor:
    return t / t.norm(dim=-1, keepdim=True) * scale


def _recurrence_inputs(r: _Rand, T, Hk, Hv, Dk, Dv, dtype) -> dict:
    """Keys of unit length, queries scaled by 1/sqrt(Dk), values ~ N(0, 1)."""
    return dict(q=_unit(r.normal(T, Hk, Dk), Dk ** -0.5).to(dtype), k=_unit(r.normal(T, Hk, Dk)).to(dtype),
                v=r.normal(T, Hv, Dv, dtype=dtype))


def _quantized(r: _Rand, n: int, k: int, mode: str, bits: int, group: int) -> dict:
    if mode == "mxfp8":
        codes = r.normal(n, k, scale=32.0).to(torch.float8_e4m3fn).view(torch.uint8).reshape(n, k // 4, 4)
        shift = torch.arange(0, 32, 8, device=DEV, dtype=torch.int32)
        weight = (codes.to(torch.int32) << shift).sum(-1, dtype=torch.int64)
        weight = torch.where(weight >= 2 ** 31, weight - 2 ** 32, weight).to(torch.int32)
    else:
        weight = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k * bits // 32), generator=r.g, device=DEV,
                               dtype=torch.int32)
    groups = k // group
    if mode == "affine":
        step = 0.12 / 2 ** bits  # weights of about +- 0.06 whatever the width
        scales = r.uniform(0.5 * step, 1.5 * step, n, groups).to(torch.bfloat16)
        biases = (-scales.float() * 2 ** (bits - 1) * r.uniform(0.9, 1.1, n, groups)).to(torch.bfloat16)
        return dict(weight=weight, scales=scales, biases=biases)
    low, high = {"mxfp4": (119, 123), "mxfp8": (114, 118), "nvfp4": (8, 24)}[mode]
    scales = torch.randint(low, high, (n, groups), generator=r.g, device=DEV, dtype=torch.int32).to(torch.uint8)
    return dict(weight=weight, scales=scales)


def _layer(r: _Rand, dims, hidden: int):
    """A layer with 4-bit group-64 projections; its weights and parameters
    beside it."""
    scheme = gdn.QuantScheme(4, 64)
    shapes = dict(qkv=(dims.conv_dim, hidden), z=(dims.value_dim, hidden), a=(dims.num_value_heads, hidden),
                  b=(dims.num_value_heads, hidden), out=(hidden, dims.value_dim))
    w = {name: _quantized(r, n, k, "affine", 4, 64) for name, (n, k) in shapes.items()}
    p = _layer_params(r, dims)
    lw = {name: gdn.LinearWeights(t, scheme) for name, t in w.items()}
    layer = gdn.Qwen3_5LinearAttention(dims, lw["qkv"], lw["z"], lw["a"], lw["b"], p["conv_w"][:, :, None],
                                       p["A_log"], p["dt_bias"], p["norm_w"], lw["out"], rms_norm_eps=EPS)
    return layer, w, p


def _pool(r: _Rand, dims, size: int, dtype):
    pool = gdn.RecurrentStatePool(size, CONV_K, dims.conv_dim, dims.num_value_heads, dims.value_head_dim,
                                  dims.key_head_dim, dtype=dtype, device=DEV)
    pool.ssm_state.normal_(0, 0.05, generator=r.g)
    pool.conv_buf[:size].copy_(r.normal(size, CONV_K - 1, dims.conv_dim, dtype=dtype))
    return pool


def _dense_layer(case, r: _Rand):
    dims = _dims(case)
    p = _layer_params(r, dims)
    none = torch.empty(0, device=DEV)  # the core uses no projection
    layer = gdn.Qwen3_5LinearAttention(dims, none, none, none, none, p["conv_w"][:, :, None], p["A_log"],
                                       p["dt_bias"], p["norm_w"], none, rms_norm_eps=EPS)
    return layer, p


def prepare(case: dict, seed: int) -> dict:
    r = _Rand(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "decode":
        dims, act = _dims(case), ACT[case["act"]]
        B, P, Hv = case["batch"], case["pool"], case["value_heads"]
        s.update(dims=dims, **_layer_params(r, dims), qkv=r.normal(B, dims.conv_dim, dtype=act),
                 a=r.normal(B, Hv, dtype=act), b=r.normal(B, Hv, dtype=act),
                 z=r.normal(B, Hv, 128, dtype=act) if case["norm"] else None)
        if P:
            s["pool"] = _pool(r, dims, P, act)
            s["slots"] = r.py.sample(range(P), B)
            s["slot_t"] = s["pool"].device_slots(s["slots"])
        else:
            s.update(conv=r.normal(B, CONV_K - 1, dims.conv_dim, dtype=act), ssm=r.normal(B, Hv, 128, 128, scale=0.05))
        return s
    if kind == "update":
        lens, Hv, dt = _lens(case), case["value_heads"], ACT[case["dtype"]]
        T = sum(lens)
        s.update(_recurrence_inputs(r, T, 16, Hv, 128, 128, dt), a=r.normal(T, Hv, dtype=dt),
                 b=r.normal(T, Hv, dtype=dt), **_gate_params(r, Hv),
                 state=r.normal(len(lens), Hv, 128, 128, scale=0.05) if case["state"] else None)
        if case["packed"]:
            s["offsets"] = _offsets(lens)
        else:
            s.update({n: s[n].reshape(len(lens), lens[0], *s[n].shape[1:]) for n in ("q", "k", "v", "a", "b")})
        return s
    if kind == "scan":
        L, Hv, dt = case["tokens"], case["value_heads"], ACT[case["dtype"]]
        s.update(_recurrence_inputs(r, L, case["key_heads"], Hv, case["key_dim"], case["value_dim"], dt),
                 g=r.uniform(0.7, 1.0, L, Hv), beta=r.uniform(0.0, 1.0, L, Hv).to(dt),
                 state=r.normal(Hv, case["value_dim"], case["key_dim"], scale=0.05))
        return s
    if kind == "core":
        lens, Hv, act = _lens(case), case["value_heads"], ACT[case["act"]]
        T, dims = sum(lens), _dims(case)
        layer, p = _dense_layer(case, r)
        s.update(dims=dims, layer=layer, **p, qkv=r.normal(T, dims.conv_dim, dtype=act),
                 z=r.normal(T, Hv, 128, dtype=act), a=r.normal(T, Hv, dtype=act), b=r.normal(T, Hv, dtype=act),
                 conv=r.normal(len(lens), CONV_K - 1, dims.conv_dim, dtype=act),
                 ssm=r.normal(len(lens), Hv, 128, 128, scale=0.05),
                 offsets=_offsets(lens) if len(lens) > 1 else None)
        return s
    if kind == "linear":
        s.update(x=r.normal(case["rows"], case["hidden"], dtype=ACT[case["act"]]),
                 scheme=gdn.QuantScheme(case["bits"], case["group"], case["mode"]),
                 w=_quantized(r, case["out"], case["hidden"], case["mode"], case["bits"], case["group"]))
        return s
    dims, act = _dims(case), ACT[case["act"]]
    layer, w, p = _layer(r, dims, case["hidden"])
    s.update(dims=dims, layer=layer, w=w, **p)
    if kind == "layer_decode":
        s["pool"] = _pool(r, dims, case["pool"], act)
        s["slots"] = r.py.sample(range(case["pool"]), case["batch"])
        s["x"] = r.normal(case["batch"], case["hidden"], dtype=act)
        s["graph"] = gdn.DecodeGraph(layer, s["pool"], s["slots"], s["x"])
    else:
        s["cache"] = layer.new_cache(act)
        s["x"] = r.normal(case["tokens"], case["hidden"], dtype=act)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(s: dict):
    kind = s["case"]["kind"]
    if kind == "decode":
        args = (s["conv_w"], s["A_log"], s["dt_bias"], s["norm_w"], EPS, s["dims"])
        if "pool" not in s:
            return gdn.fused_decode_step(s["qkv"], s["z"], s["a"], s["b"], s["conv"], s["ssm"], *args)
        pool = s["pool"]
        out, conv, ssm = gdn.fused_decode_step(s["qkv"], s["z"], s["a"], s["b"], pool.conv_buf, pool.ssm_state,
                                               *args, slots=s["slot_t"], conv_half=pool.conv_half_dev,
                                               conv_arrivals=pool.conv_arrivals)
        pool.advance(s["slots"], s["slot_t"], device_flipped=True)
        return out, conv, ssm
    if kind == "update":
        return gdn.gated_delta_update(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"], s["state"],
                                      cu_seqlens=s.get("offsets"))
    if kind == "scan":
        return gdn.gated_delta_scan(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"])
    if kind == "core":
        return s["layer"].core(s["qkv"], s["z"], s["a"], s["b"], s["conv"], s["ssm"], s["offsets"])
    if kind == "linear":
        return gdn.quantized_linear(s["x"], s["w"], s["scheme"])
    if kind == "layer_decode":
        out = s["graph"].step(s["x"])
        return out, s["pool"].conv_buf, s["pool"].ssm_state
    cache = copy.copy(s["cache"])  # the call replaces the cache's tensors; the prompt starts anew each pass
    out = s["layer"](s["x"], cache)
    return (out, *cache.state())


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _weight_bytes(n: int, k: int, mode: str, bits: int, group: int) -> int:
    per_group = 4 if mode == "affine" else 1
    return n * k * bits // 8 + n * (k // group) * per_group


def _recurrent_bytes(tokens: int, runs: int, dims, es: int, y: int) -> int:
    """qkv, a, b (and z) in, y out at ``y`` bytes a value, states in and out."""
    per_token = (dims.conv_dim + 2 * dims.num_value_heads) * es + dims.value_dim * y
    return tokens * per_token + runs * dims.num_value_heads * 128 * 128 * 8


def _step_flops(tokens: int, dims) -> int:
    """Decay, two products with the state and the rank-1 update."""
    return tokens * dims.num_value_heads * 7 * 128 * 128


def _chunk_flops(tokens: int, dims) -> int:
    """The chunk form's products: K K^T, Q K^T, Tb R, P D and the inverse over
    64 tokens, and three with the 128 x 128 state."""
    return tokens * dims.num_value_heads * (10 * CHUNK * 128 + 6 * 128 * 128)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "scan":
        L, Hk, Hv, Dk, Dv = (case[n] for n in ("tokens", "key_heads", "value_heads", "key_dim", "value_dim"))
        es = 2 if case["dtype"] == "bf16" else 4
        return dict(bytes=L * (2 * Hk * Dk * es + Hv * Dv * (es + 4) + Hv * (4 + es)) + 8 * Hv * Dk * Dv,
                    flops=L * Hv * 7 * Dk * Dv)
    if kind == "linear":
        m, n, k = case["rows"], case["out"], case["hidden"]
        es = 2 if case["act"] == "bf16" else 4
        return dict(bytes=_weight_bytes(n, k, case["mode"], case["bits"], case["group"]) + m * (n + k) * es,
                    flops=2 * m * n * k)
    dims = _dims(case)
    es = 2 if case.get("act", case.get("dtype")) == "bf16" else 4
    if kind == "update":
        T = sum(_lens(case))
        return dict(bytes=_recurrent_bytes(T, case["runs"], dims, es, 4)
                    - (0 if case["state"] else case["runs"] * dims.num_value_heads * 128 * 128 * 4),
                    flops=_chunk_flops(T, dims))
    conv = 2 * (CONV_K - 1) * dims.conv_dim * es  # a run's conv state in and out
    if kind == "core":
        T = sum(_lens(case))
        return dict(bytes=_recurrent_bytes(T, case["runs"], dims, es, 2 * es) + case["runs"] * conv,
                    flops=_chunk_flops(T, dims))
    if kind == "decode":
        B = case["batch"]
        return dict(bytes=_recurrent_bytes(B, B, dims, es, 2 * es if case["norm"] else 4) + B * conv
                    + dims.conv_dim * CONV_K * 4, flops=_step_flops(B, dims))
    hidden = case["hidden"]
    rows = case["batch"] if kind == "layer_decode" else case["tokens"]
    n_in = dims.conv_dim + dims.value_dim + 2 * dims.num_value_heads
    runs = rows if kind == "layer_decode" else 1
    weights = _weight_bytes(n_in, hidden, "affine", 4, 64) + _weight_bytes(hidden, dims.value_dim, "affine", 4, 64)
    flops = 2 * rows * hidden * (n_in + dims.value_dim)
    flops += _step_flops(rows, dims) if kind == "layer_decode" else _chunk_flops(rows, dims)
    return dict(bytes=weights + 2 * rows * hidden * es + runs * (conv + dims.num_value_heads * 128 * 128 * 8),
                flops=flops)


def tolerance(case: dict) -> dict:
    """About four times the difference measured between each path and float64
    on the same inputs: bf16 results carry one rounding (2e-3), or those of
    the layer's chain with weights rounded to bf16 (7e-3); the chunked
    prompts' bf16 hi + lo operands give 5e-6 to 2e-5, float32 products 1e-6
    (5e-6 where x enters as bf16 hi + lo), the scan 1e-7."""
    kind = case["kind"]
    bf16 = case.get("act") == "bf16"
    if kind == "linear":
        return {"rel": 8e-3, "max": 5e-2} if bf16 else {"rel": 2e-5, "max": 5e-4}
    if kind == "scan":
        return {"rel": 1e-6, "max": 5e-5}
    if kind == "update":
        return {"rel": 5e-5, "max": 2e-3}
    if bf16 and (kind == "layer_prompt" or kind == "layer_decode" and case["batch"] > 64):
        return {"rel": 2.5e-2, "max": 2e-1}
    if bf16 and (kind != "decode" or case["norm"]):
        return {"rel": 8e-3, "max": 5e-2}
    return {"rel": 1e-5, "max": 5e-4} if kind == "decode" else {"rel": 8e-5, "max": 2e-3}


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------


def _round(t: torch.Tensor, dtype) -> torch.Tensor:
    """Held in ``dtype`` where the reference's layer holds it there."""
    return t.to(dtype).double()


def _silu64(t):
    return t * torch.sigmoid(t)


def _gates64(a, b, A_log, dt_bias):
    g = torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(a.double() + dt_bias.double()))
    return g, _round(torch.sigmoid(b.double()), b.dtype)


def _recurrence64(q, k, v, g, beta, state, lens):
    """The recurrence over packed runs, all runs' tokens t at once. q, k
    (T, Hk, Dk), v (T, Hv, Dv), g, beta (T, Hv), state (N, Hv, Dv, Dk)."""
    rep = v.shape[1] // q.shape[1]
    order = sorted(range(len(lens)), key=lambda i: -lens[i])
    first = torch.tensor([_offsets(lens)[i] for i in order], device=DEV)
    S = state.double()[order].contiguous()
    g, beta = g.double(), beta.double()
    y = torch.zeros(v.shape, dtype=torch.float64, device=DEV)
    n = len(order)
    for t in range(max(lens)):
        while lens[order[n - 1]] <= t:
            n -= 1
        rows = first[:n] + t
        kt = k[rows].double().repeat_interleave(rep, dim=1)
        qt = q[rows].double().repeat_interleave(rep, dim=1)
        St = S[:n]
        St *= g[rows][:, :, None, None]
        delta = (v[rows].double() - (St * kt[:, :, None, :]).sum(-1)) * beta[rows][:, :, None]
        St.addcmul_(delta[..., None], kt[:, :, None, :])
        y[rows] = (St * qt[:, :, None, :]).sum(-1)
    out = torch.empty_like(S)
    out[order] = S
    return y, out


def _front64(qkv, conv, conv_w, dims, act, lens):
    """Conv over each run's (state, tokens), SiLU, and the scaled norms of q
    and k; the results rounded to the activations' type as the layer does."""
    q, k, v, new = [], [], [], []
    Hk, key = dims.num_key_heads, dims.key_dim
    w = conv_w.double()
    inv = _round(torch.tensor(128 ** -0.5, dtype=torch.float64), act)
    inv2 = _round(torch.tensor(1 / 128, dtype=torch.float64), act)
    for i, (t0, n) in enumerate(zip(_offsets(lens), lens)):
        x = torch.cat([conv[i].double(), qkv[t0:t0 + n].double()])
        new.append(x[-(CONV_K - 1):])
        o = _round(sum(w[:, j] * x[j:j + n] for j in range(CONV_K)), act)
        o = _round(_silu64(o), act)
        heads = o[:, :2 * key].reshape(n, 2 * Hk, 128)
        heads = _round(heads * torch.rsqrt(heads.square().mean(-1, keepdim=True) + 1e-6), act)
        q.append(_round(heads[:, :Hk] * inv2.item(), act))
        k.append(_round(heads[:, Hk:] * inv.item(), act))
        v.append(o[:, 2 * key:].reshape(n, dims.num_value_heads, 128))
    return torch.cat(q), torch.cat(k), torch.cat(v), torch.stack(new)


def _norm64(y, z, norm_w, act):
    x = _round(y, act)
    x = _round(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * norm_w.double(), act)
    return _silu64(z.double()) * x


def _core64(s, qkv, z, a, b, conv, ssm, lens, act):
    q, k, v, new_conv = _front64(qkv, conv, s["conv_w"], s["dims"], act, lens)
    g, beta = _gates64(a, b, s["A_log"], s["dt_bias"])
    y, new_ssm = _recurrence64(q, k, v, g, beta, ssm, lens)
    return (y if z is None else _norm64(y, z, s["norm_w"], act)), new_conv, new_ssm


def _weight64(w: dict, mode: str, bits: int, group: int) -> torch.Tensor:
    n, words = w["weight"].shape
    k = words * 32 // bits
    stream = torch.cat([w["weight"].long() & 0xFFFFFFFF, torch.zeros(n, 1, dtype=torch.int64, device=DEV)], dim=1)
    at = torch.arange(k, device=DEV) * bits
    word, shift = at // 32, at % 32
    codes = ((stream[:, word] >> shift) | (stream[:, word + 1] << (32 - shift))) & (2 ** bits - 1)
    if mode == "affine":
        rep = lambda t: t.double().repeat_interleave(group, dim=1)
        return codes * rep(w["scales"]) + rep(w["biases"])
    if bits == 8:
        values = codes.to(torch.uint8).view(torch.float8_e4m3fn).double()
    else:
        e2m1 = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=DEV)
        values = torch.cat([e2m1, -e2m1])[codes]
    if mode == "nvfp4":
        scale = w["scales"].view(torch.float8_e4m3fn).double()
    else:
        scale = torch.exp2(w["scales"].double() - 127)
    return values * scale.repeat_interleave(group, dim=1)


def _layer64(s, x, conv, ssm, lens, act):
    proj = lambda name: _round(x.double() @ _weight64(s["w"][name], "affine", 4, 64).T, act).to(act)
    T, Hv = x.shape[0], s["dims"].num_value_heads
    z = proj("z").reshape(T, Hv, 128)
    out, new_conv, new_ssm = _core64(s, proj("qkv"), z, proj("a"), proj("b"), conv, ssm, lens, act)
    out = _round(out, act).reshape(T, -1) @ _weight64(s["w"]["out"], "affine", 4, 64).T
    return out, new_conv, new_ssm


def _pool64(s, step):
    """A step of a pool's slots, all at their first halves: the other halves
    receive the rolled rows, the slots their states."""
    pool, slots = s["pool"], s["slots"]
    out, new_conv, new_ssm = step(pool.conv_buf[slots], pool.ssm_state[slots])
    conv, ssm = pool.conv_buf.double(), pool.ssm_state.double()
    conv[[i + pool.batch for i in slots]] = new_conv
    ssm[slots] = new_ssm
    return out, conv, ssm


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "decode":
        act, ones = ACT[case["act"]], [1] * case["batch"]
        step = lambda conv, ssm: _core64(s, s["qkv"], s["z"], s["a"], s["b"], conv, ssm, ones, act)
        return _pool64(s, step) if "pool" in s else step(s["conv"], s["ssm"])
    if kind == "update":
        lens = _lens(case)
        flat = {n: s[n].reshape(sum(lens), *s[n].shape[(1 if case["packed"] else 2):]) for n in ("q", "k", "v", "a", "b")}
        g, beta = _gates64(flat["a"], flat["b"], s["A_log"], s["dt_bias"])
        state = s["state"]
        if state is None:
            state = torch.zeros(len(lens), case["value_heads"], 128, 128, device=DEV)
        y, state = _recurrence64(flat["q"], flat["k"], flat["v"], g, beta, state, lens)
        return y.reshape(s["v"].shape), state
    if kind == "scan":
        y, state = _recurrence64(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"][None], [case["tokens"]])
        return y, state[0]
    if kind == "core":
        out, conv, ssm = _core64(s, s["qkv"], s["z"], s["a"], s["b"], s["conv"], s["ssm"], _lens(case), ACT[case["act"]])
        return out.reshape(out.shape[0], -1), conv, ssm
    if kind == "linear":
        return s["x"].double() @ _weight64(s["w"], case["mode"], case["bits"], case["group"]).T
    if kind == "layer_decode":
        return _pool64(s, lambda conv, ssm: _layer64(s, s["x"], conv, ssm, [1] * case["batch"], ACT[case["act"]]))
    conv, ssm = s["cache"].state()
    out, conv, ssm = _layer64(s, s["x"], conv[None], ssm[None], [case["tokens"]], ACT[case["act"]])
    return out, conv[0], ssm[0]
