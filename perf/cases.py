"""The work that users of this framework have it do, as timed and compared cases.

Kinds of case, each through the entry points a program calls:

* ``linear``: one row through one N:M-sparse Linear, called eagerly: fp16
  through the module (`NmSparseLinear`, what a swapped model calls), bf16 and
  fp32 through the wrapper (`nmsparse_spmv_forward_hip`).
* ``rows``: several rows through one sparse Linear without a dense weight,
  called eagerly (a prompt or a batch): fp16 through the module, bf16 through
  `nmsparse_spmm_forward_hip`.
* ``mlp``: a SwiGLU MLP on the rows of a serving batch (gate and up of one
  input, down on their SiLU product), captured in a hipGraph as a serving loop
  of a fixed batch size keeps it.
* ``step``: one decode step of a swapped decoder at a position of a filled
  cache, captured in a hipGraph and replayed (the fixed-context protocol of
  the benchmark); returns the logits and the updated caches.
* ``prefill``: a whole prompt in one `Decoder.prefill` pass, called eagerly;
  returns the last position's logits and the filled caches.

Sizes are those of the repository's Llama-3.1 and Qwen3 configurations and
odd ones beside them; weights N(0, 1/K) with one seeded mask per matrix.
"""
from __future__ import annotations

import dataclasses
import math

import torch

from spmv_decode_amd import NmSparseLinear
from spmv_decode_amd.decode.model import CONFIGS, Decoder, project_rows_group, project_rows_silu_mul
from spmv_decode_amd.decode.runner import cache_length
from spmv_decode_amd.hip_spmv import nmsparse_spmm_forward_hip, nmsparse_spmv_forward_hip
from spmv_decode_amd.nmsparse_linear import tie_siblings

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # The smallest call: a key projection of the smallest decoder, one row, latency only.
        dict(name="linear_small", kind="linear", K=1024, h=1024, M=64, dtype="fp16"),
        # A wide projection in bf16 at 2:4 with sizes that fill no tile evenly.
        dict(name="linear_bf16_ragged", kind="linear", K=5004, h=17280, M=4, dtype="bf16"),
        # A down projection kept in fp32.
        dict(name="linear_fp32", kind="linear", K=14336, h=4096, M=32, dtype="fp32"),
        # Batched decode of a few sequences: every weight read once for 4 rows.
        dict(name="mlp_batch4", kind="mlp", dim=4096, inter=14336, M=64, rows=4, dtype="fp16"),
        # A serving batch past the small-batch kernel, bf16, an odd row count.
        dict(name="mlp_batch33", kind="mlp", dim=5120, inter=17408, M=16, rows=33, dtype="bf16"),
        # A prefill chunk of 128 rows.
        dict(name="mlp_batch128", kind="mlp", dim=4096, inter=14336, M=64, rows=128, dtype="fp16"),
        # A prompt through a sparse-only Linear: more rows than one kernel tile, unevenly.
        dict(name="rows_200", kind="rows", K=14336, h=4096, M=64, rows=200, dtype="fp16"),
        # A long prompt: compute-bound, the largest single product.
        dict(name="rows_2048", kind="rows", K=5120, h=25600, M=32, rows=2048, dtype="bf16"),
        # The benchmark's decode step.
        dict(name="step_llama_512", kind="step", model="llama-3.1-8b", layers=32, M=64, ctx=512),
        # A small model's decode step: launches and latency.
        dict(name="step_qwen06b_100", kind="step", model="qwen3-0.6b", layers=28, M=32, ctx=100),
        # A few layers far into a long context: the caches weigh as much as the weights.
        dict(name="step_qwen14b_4001", kind="step", model="qwen3-14b", layers=8, M=16, ctx=4001),
        # A whole prompt of the benchmark's model.
        dict(name="prefill_llama_500", kind="prefill", model="llama-3.1-8b", layers=32, M=64, P=500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "rows", "mlp", "mlp", "step", "step", "prefill"])
    M = rng.choice([4, 8, 16, 32, 64, 128, 256])
    if kind in ("linear", "rows"):
        K = max(1, round(_log_int(rng, 512, 25600) / M)) * M
        h = max(1, round(_log_int(rng, 512, 25600) / 128)) * 128
        if kind == "linear":
            return dict(kind=kind, K=K, h=h, M=M, dtype=rng.choice(["fp16", "bf16", "fp32"]))
        return dict(kind=kind, K=K, h=h, M=M, rows=_log_int(rng, 2, 2048), dtype=rng.choice(["fp16", "bf16"]))
    if kind == "mlp":
        dim = rng.choice([1024, 2048, 3072, 4096, 5120])
        inter = max(2, round(dim * rng.uniform(2.5, 5.0) / 256)) * 256
        return dict(kind=kind, dim=dim, inter=inter, M=M, rows=_log_int(rng, 2, 400),
                    dtype=rng.choice(["fp16", "bf16"]))
    model = rng.choice(["qwen3-0.6b", "llama-3.1-8b", "qwen3-14b"])
    layers = rng.randint(1, 6)
    if kind == "step":
        return dict(kind=kind, model=model, layers=layers, M=M, ctx=_log_int(rng, 12, 6000))
    return dict(kind=kind, model=model, layers=layers, M=M, P=_log_int(rng, 5, 1500))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(gen, *shape, std=1.0, dtype=torch.float16):
    return (torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float32) * std).to(dtype)


def _packed(gen, K, h, M, dtype=torch.float16):
    """Packed weights [K/2, h] and in-group positions [K/M, M/2] of one M/2:M Linear."""
    mi = torch.rand(K // M, M, generator=gen, device=DEV).argsort(dim=1)[:, :M // 2].sort(dim=1).values
    return _normal(gen, K // 2, h, std=K ** -0.5, dtype=dtype), mi.to(torch.uint8).contiguous()


def _linear(gen, K, h, M, dtype=torch.float16):
    lin = NmSparseLinear.empty(h, K, M, DEV, dtype=dtype)
    lin.mat_data, lin.mat_index = _packed(gen, K, h, M, dtype)
    return lin


def _config(case):
    return dataclasses.replace(CONFIGS[case["model"]], n_layers=case["layers"])


def _decoder(cfg, M, gen):
    """A decoder as swap_to_nmsparse leaves one without dense weights, every value drawn from `gen`."""
    with torch.device("meta"):
        model = Decoder(cfg)
    for blk in model.layers:
        for sub in (blk.self_attn, blk.mlp):
            for name, mod in list(sub.named_children()):
                if isinstance(mod, torch.nn.Linear):
                    setattr(sub, name, _linear(gen, mod.in_features, mod.out_features, M))
        at, mlp = blk.self_attn, blk.mlp
        tie_siblings(at.q_proj, at.k_proj, at.v_proj)
        tie_siblings(mlp.gate_proj, mlp.up_proj)
    for mod in model.modules():
        for name, par in list(mod.named_parameters(recurse=False)):
            if par.ndim == 1:
                val = 1.0 + _normal(gen, *par.shape, std=0.1)
            else:
                val = _normal(gen, *par.shape, std=0.02)
            setattr(mod, name, torch.nn.Parameter(val, requires_grad=False))
    return model


def _fill_cache(model, gen, n):
    """n cached positions of every layer, at the scale of the keys and values these weights give."""
    hd = model.cfg.head_dim
    for k, v in zip(model.k_cache_t, model.v_cache_t):
        k[:, :hd, :n] = _normal(gen, *k[:, :hd, :n].shape)
        v[:, :, :n] = _normal(gen, *v[:, :, :n].shape)


def _captured(fn):
    """fn() recorded in a hipGraph after a warm-up on the capture stream: (graph, its outputs)."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream), torch.no_grad():
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream), torch.no_grad():
        out = fn()
    return graph, out


def _inputs(case, seed):
    """Everything that is drawn for a case: its weights or model, then its activations."""
    gen = _generator(seed)
    if case["kind"] in ("linear", "rows"):
        dt = DTYPES[case["dtype"]]
        lin = _linear(gen, case["K"], case["h"], case["M"], dt)
        return dict(lin=lin, x=_normal(gen, 1, case.get("rows", 1), case["K"], dtype=dt))
    if case["kind"] == "mlp":
        dt, dim, inter, M = DTYPES[case["dtype"]], case["dim"], case["inter"], case["M"]
        gate, up, down = (_linear(gen, K, h, M, dt) for K, h in ((dim, inter), (dim, inter), (inter, dim)))
        return dict(gate=gate, up=up, down=down, x=_normal(gen, case["rows"], dim, dtype=dt))
    cfg = _config(case)
    model = _decoder(cfg, case["M"], gen)
    if case["kind"] == "step":
        model.setup_cache(cache_length(case["ctx"] + 1), torch.device(DEV))
        _fill_cache(model, gen, case["ctx"])
        n = 1
    else:
        model.setup_cache(cache_length(case["P"] + 1), torch.device(DEV))
        n = case["P"]
    return dict(model=model, ids=torch.randint(0, cfg.vocab, (n,), generator=gen, device=DEV))


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"], s["dtype"] = case["kind"], case.get("dtype")
    if case["kind"] == "mlp":
        x, gate, up, down = s["x"], s["gate"], s["up"], s["down"]
        s["graph"], s["out"] = _captured(lambda: project_rows_silu_mul(down, *project_rows_group((gate, up), x)))
    elif case["kind"] == "step":
        model, token = s["model"], s["ids"].view(1, 1)
        pos = torch.full((1,), case["ctx"], dtype=torch.long, device=DEV)
        s["pos"] = pos
        s["graph"], s["out"] = _captured(lambda: model.forward_step(token, pos))
    return s


def _caches(model):
    return {"k": model.k_store[:, :, :model.cfg.head_dim], "v": list(model.v_cache_t)}


def run(s):
    if "graph" in s:
        s["graph"].replay()
        return {"logits": s["out"], **_caches(s["model"])} if s["kind"] == "step" else s["out"]
    with torch.no_grad():
        if s["kind"] == "prefill":
            return {"logits": s["model"].prefill(s["ids"]), **_caches(s["model"])}
        lin, x = s["lin"], s["x"]
        if s["dtype"] == "fp16":
            return lin(x)
        if s["kind"] == "linear":
            return nmsparse_spmv_forward_hip(x[0], lin.mat_data, lin.mat_index, lin.w, lin.h, lin.block_width, 128,
                                             lin.vec_width, 1, x.shape[-1])
        return nmsparse_spmm_forward_hip(x, lin.mat_data, lin.mat_index, lin.w, lin.h, lin.block_width, lin.vec_width)


# --------------------------------------------------------------------------
# What a pass cannot do without, and how exact its results are
# --------------------------------------------------------------------------
def _layer_shapes(cfg):
    qd, kvd = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    return [(cfg.dim, qd), (cfg.dim, kvd), (cfg.dim, kvd), (qd, cfg.dim), (cfg.dim, cfg.inter), (cfg.dim, cfg.inter),
            (cfg.inter, cfg.dim)]


def work(case):
    kind = case["kind"]
    if kind in ("linear", "rows"):
        e, R, K, h = 4 if case["dtype"] == "fp32" else 2, case.get("rows", 1), case["K"], case["h"]
        w = K // 2
        return {"bytes": e * (w * h + R * K + R * h) + w, "flops": 2 * R * w * h}
    if kind == "mlp":
        dim, inter, R = case["dim"], case["inter"], case["rows"]
        weights = 3 * (dim // 2) * inter
        return {"bytes": 2 * weights + dim + inter // 2 + 4 * R * dim, "flops": 2 * R * weights}
    cfg = _config(case)
    weights = cfg.n_layers * sum((K // 2) * h for K, h in _layer_shapes(cfg))
    head = cfg.vocab * cfg.dim
    kv = cfg.n_layers * 2 * cfg.n_kv_heads * cfg.head_dim  # cached values per position
    n = 1 if kind == "step" else case["P"]
    seen = case["ctx"] + 1 if kind == "step" else (n + 1) / 2  # positions a query attends to, on average
    read = kv * case["ctx"] if kind == "step" else 0
    attention = 4 * n * seen * cfg.n_layers * cfg.n_heads * cfg.head_dim
    return {"bytes": 2 * (weights + head + read + kv * n + n * cfg.dim + cfg.vocab),
            "flops": 2 * n * weights + 2 * head + attention}


def tolerance(case):
    """About four times the distance from 64 bits measured on an MI355X: one
    rounding to the type for a product (2.2e-4 in fp16, 1.7e-3 in bf16, sums
    in fp32 1.7e-7), two chained ones for an MLP (4.4e-4, 3.5e-3); a model's
    roundings layer after layer (a step 1.0e-3 to 3.9e-3, and 3.3e-3 from one
    run to the next; a prompt 1.5e-3)."""
    kind = case["kind"]
    if kind in ("linear", "rows"):
        return {"rel": {"fp16": 1e-3, "bf16": 7e-3, "fp32": 1e-6}[case["dtype"]]}
    if kind == "mlp":
        return {"rel": {"fp16": 1.8e-3, "bf16": 1.4e-2}[case["dtype"]]}
    return {"rel": 1.4e-2 if kind == "step" else 6e-3, "max": 0.3}


# --------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------
def _product(x, lin):
    """x [rows, K] (64 bits) times the packed weights."""
    groups, nnz = lin.mat_index.shape
    M = x.shape[-1] // groups
    pos = (torch.arange(groups, device=DEV)[:, None] * M + lin.mat_index.long()).view(-1)
    y = x[:, pos]
    md = lin.mat_data
    return torch.cat([y @ part.double() for part in md.split(4096, dim=1)], dim=1)


def _silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _angles(cfg, positions):
    inv = cfg.rope_theta ** (-torch.arange(0, cfg.head_dim, 2, device=DEV).double() / cfg.head_dim)
    sc = cfg.rope_scaling
    if sc:  # low frequencies divided by the factor, high ones kept, a linear blend between
        turns = sc["original_max_position_embeddings"] * inv / (2 * math.pi)
        blend = ((turns - sc["low_freq_factor"]) / (sc["high_freq_factor"] - sc["low_freq_factor"])).clamp(0, 1)
        inv = (1 - blend) * inv / sc["factor"] + blend * inv
    return positions.double()[:, None] * inv


def _turn(x, ang):
    """Rotary embedding of [n, heads, d] on (even, odd) pairs."""
    a, b = x[..., 0::2], x[..., 1::2]
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    return torch.stack((a * c - b * s, a * s + b * c), dim=-1).flatten(-2)


def _exact_model(model, ids, start):
    """Tokens `ids` at positions start.. of the model's caches: (logits of the last, keys, values)."""
    cfg, n = model.cfg, ids.numel()
    hd, kvh, g = cfg.head_dim, cfg.n_kv_heads, cfg.n_heads // cfg.n_kv_heads
    end = start + n
    ang = _angles(cfg, torch.arange(start, end, device=DEV))
    hidden = torch.arange(end, device=DEV)[None, :] > torch.arange(start, end, device=DEV)[:, None]
    x = model.embed_tokens.weight[ids].double()
    keys, values = model.k_store[:, :, :hd].double(), [v.double() for v in model.v_cache_t]
    for i, blk in enumerate(model.layers):
        at, mlp = blk.self_attn, blk.mlp
        y = _rms(x, blk.input_layernorm.weight, cfg.norm_eps)
        q, k, v = (_product(y, p).view(n, -1, hd) for p in (at.q_proj, at.k_proj, at.v_proj))
        if cfg.qk_norm:
            q, k = _rms(q, at.q_norm.weight, cfg.norm_eps), _rms(k, at.k_norm.weight, cfg.norm_eps)
        keys[i, :, :, start:end] = _turn(k, ang).permute(1, 2, 0)
        values[i][:, :, start:end] = v.permute(1, 2, 0)
        heads = []
        for j in range(kvh):  # [g * n, d] queries of one key/value head
            qj = _turn(q, ang)[:, j * g:(j + 1) * g].transpose(0, 1).reshape(g * n, hd)
            p = qj @ keys[i, j, :, :end] / math.sqrt(hd)
            p = torch.softmax(p.masked_fill(hidden.repeat(g, 1), -math.inf), dim=-1)
            heads.append((p @ values[i][j, :, :end].t().contiguous()).view(g, n, hd))
        y = torch.cat(heads).transpose(0, 1).reshape(n, -1)
        x = x + _product(y, at.o_proj)
        y = _rms(x, blk.post_attention_layernorm.weight, cfg.norm_eps)
        x = x + _product(_silu_mul(_product(y, mlp.gate_proj), _product(y, mlp.up_proj)), mlp.down_proj)
    last = _rms(x[-1:], model.norm.weight, cfg.norm_eps)
    logits = torch.cat([last @ part.double().t() for part in model.lm_head.weight.split(16384)], dim=1)
    return {"logits": logits, "k": keys, "v": values}


def exact(case, seed):
    s = _inputs(case, seed)
    with torch.no_grad():
        if case["kind"] in ("linear", "rows"):
            y = _product(s["x"][0].double(), s["lin"])
            return y if case["kind"] == "linear" and case["dtype"] != "fp16" else y[None]
        if case["kind"] == "mlp":
            x = s["x"].double()
            return _product(_silu_mul(_product(x, s["gate"]), _product(x, s["up"])), s["down"])
        return _exact_model(s["model"], s["ids"], case.get("ctx", 0))
