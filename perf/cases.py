"""The work a program has this library do, as timed cases.

Each case is one pass through the public entry points over one kind of call,
for the Qwen3.6 full-attention layers (16 query heads, 2 KV heads, head_dim
256, f16 cache):

  token    one generated token through `layers` layers: Engine.forward_proj
           (from the f32 projections) or Engine.forward (from f16 q / k / v)
  verify   the draft tokens of speculative decoding after a long context:
           attn_verify
  prompt   n prompt tokens through one layer: Engine.forward_batched_proj or
           Engine.forward_batched, on an empty cache or after `past` rows
  ragged   one token for each of many independent sequences:
           attn_decode_ragged with the caller's workspace
  oproj    the output projection of one token in `layers` layers: matvec_bf16
           or matvec_q4

Inputs are drawn N(0, 1), which is what normed queries and keys look like; the
projections are scaled up so that the norm has something to do.
"""
from __future__ import annotations

import math

import torch

import moe_infer_amd as mi

H, G, D = 16, 2, 256
Q_COLS, KV_COLS = H * D, G * D
ROPE_THETA, ROTARY, EPS = 1e7, 64, 1e-6


def listed():
    return [
        # A chat's token a few hundred rows in: the smallest call, in which
        # launches and latency are everything.
        {"name": "token_517", "kind": "token", "proj": True, "layers": 10, "pos": 517},
        # The same token at the end of a 32768-row context, layer by layer
        # from HBM.
        {"name": "token_32k", "kind": "token", "proj": False, "layers": 4, "pos": 32767},
        # Four draft tokens of the MTP head verified after 65536 rows.
        {"name": "verify_4_65536", "kind": "verify", "n": 4, "past": 65536},
        # A longer draft after a mid-length context.
        {"name": "verify_12_9001", "kind": "verify", "n": 12, "past": 9001},
        # A short question on an empty cache, from its projections.
        {"name": "prompt_333", "kind": "prompt", "proj": True, "n": 333, "past": 0},
        # A page of text on an empty cache, from its projections.
        {"name": "prompt_1900", "kind": "prompt", "proj": True, "n": 1900, "past": 0},
        # A full 4096-token prompt, from ready q / k / v.
        {"name": "prompt_4096", "kind": "prompt", "proj": False, "n": 4096, "past": 0},
        # The next chunk of a long document that is already in the cache.
        {"name": "chunk_512_16384", "kind": "prompt", "proj": False, "n": 512, "past": 16384},
        # A small serving batch of short conversations.
        {"name": "ragged_8", "kind": "ragged", "batch": 8, "lo": 100, "hi": 3000},
        # A full serving batch of long ones.
        {"name": "ragged_64", "kind": "ragged", "batch": 64, "lo": 1024, "hi": 32768},
        # The output projection behind each layer's attention, both weight
        # formats.
        {"name": "oproj_bf16", "kind": "oproj", "q4": False, "layers": 10, "out_dim": 2048,
         "in_dim": 4096, "group_size": 0},
        {"name": "oproj_q4", "kind": "oproj", "q4": True, "layers": 10, "out_dim": 2048,
         "in_dim": 4096, "group_size": 64},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("token", "token", "verify", "prompt", "prompt", "chunk", "ragged", "oproj"))
    if kind == "token":
        return {"kind": "token", "proj": rng.random() < 0.5, "layers": rng.choice((4, 10)),
                "pos": _log(rng, 1, 32767)}
    if kind == "verify":
        return {"kind": "verify", "n": rng.randint(2, 16), "past": _log(rng, 100, 65536)}
    if kind == "prompt":
        return {"kind": "prompt", "proj": rng.random() < 0.5, "n": _log(rng, 17, 4096), "past": 0}
    if kind == "chunk":
        return {"kind": "prompt", "proj": rng.random() < 0.5, "n": _log(rng, 17, 1024),
                "past": _log(rng, 100, 16384)}
    if kind == "ragged":
        batch = _log(rng, 2, 64)
        hi = _log(rng, 500, 32768)
        return {"kind": "ragged", "batch": batch, "lo": rng.randint(1, hi), "hi": hi}
    q4 = rng.random() < 0.5
    step = 2048 if q4 else 512
    return {"kind": "oproj", "q4": q4, "layers": rng.choice((4, 10)),
            "out_dim": rng.randint(1000, 4096), "in_dim": step * rng.randint(1, 8192 // step),
            "group_size": rng.choice((32, 64, 128)) if q4 else 0}


# ------------------------------------------------------------------ inputs --


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, dtype=torch.float16):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=dtype)


def _projections(gen, n):
    """f32 q_proj [n, H, 2D], k, v [n, G, D] and the bf16 norm weights."""
    f = torch.float32
    return {"qp": 3 * _normal(gen, n, H, 2 * D, dtype=f), "k": 3 * _normal(gen, n, G, D, dtype=f),
            "v": _normal(gen, n, G, D, dtype=f),
            "qw": (1 + 0.1 * _normal(gen, D, dtype=f)).bfloat16(),
            "kw": (1 + 0.1 * _normal(gen, D, dtype=f)).bfloat16()}


def _ready(gen, n):
    """f16 q, gate [n, H, D] and k, v [n, G*D]."""
    return {"q": _normal(gen, n, H, D), "k": _normal(gen, n, KV_COLS),
            "v": _normal(gen, n, KV_COLS), "gate": _normal(gen, n, H, D)}


def _layer_inputs(case, gen):
    n = case.get("n", 1)
    return _projections(gen, n) if case.get("proj") else _ready(gen, n)


def _past(gen, rows):
    return _normal(gen, rows, KV_COLS), _normal(gen, rows, KV_COLS)


def _lengths(case, seed):
    """Sequence lengths in [lo, hi] and their block-aligned first rows."""
    g = torch.Generator().manual_seed(seed)
    ln = torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=g)
    blocks = (ln + 31) // 32 * 32
    return ln, torch.cumsum(blocks, 0) - blocks, int(blocks.sum())


def _ragged_inputs(case, gen, rows):
    return {"k": _normal(gen, rows, KV_COLS), "v": _normal(gen, rows, KV_COLS),
            "q": _normal(gen, case["batch"], H, D), "gate": _normal(gen, case["batch"], H, D)}


def _weights(case, gen):
    """One layer's x and weight matrix."""
    o, i = case["out_dim"], case["in_dim"]
    x = 0.1 * _normal(gen, i)
    if not case["q4"]:
        return {"x": x, "w": (0.02 * _normal(gen, o, i, dtype=torch.float32)).bfloat16()}
    groups = i // case["group_size"]
    w = torch.randint(-2**31, 2**31, (o, i // 8), generator=gen, device="cuda",
                      dtype=torch.int64).to(torch.int32)
    scales = (0.005 * (1 + 0.2 * _normal(gen, o, groups, dtype=torch.float32))).bfloat16()
    biases = (-7.5 * scales.float()).bfloat16()
    return {"x": x, "w": w, "scales": scales, "biases": biases}


class _DeviceRows:
    """A cache buffer as torch.as_tensor takes it; the tensor holds this
    object, and this object the cache that owns the memory."""

    def __init__(self, cache, ptr, numel):
        self.cache = cache
        self.__cuda_array_interface__ = {"shape": (numel,), "typestr": "<f2",
                                         "data": (ptr, False), "version": 2}


def _cache_views(cache):
    """The K and V buffers of every layer as tensors (device layout)."""
    numel = cache.capacity * KV_COLS
    return [torch.as_tensor(_DeviceRows(cache, p, numel), device="cuda")
            for layer in cache.full_layers for p in cache.layer_ptrs(layer)]


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "ragged":
        ln, off, rows = _lengths(case, seed)
        x = _ragged_inputs(case, gen, rows)
        kb, vb = mi.kv_pack(x.pop("k"), x.pop("v"), G)
        return {"case": case, "k": kb, "v": vb, "lengths": ln.int().cuda(),
                "offsets": off.int().cuda(), "out": torch.empty_like(x["q"]),
                "workspace": mi.ragged_workspace(case["batch"], case["hi"]), **x}
    if kind == "oproj":
        return {"case": case, "layers": [_weights(case, gen) for _ in range(case["layers"])]}
    layers = case.get("layers", 1)
    past = case["pos"] if kind == "token" else case["past"]
    n = case.get("n", 1)
    cache = mi.Cache(num_layers=layers, num_q_heads=H, num_kv_heads=G, head_dim=D,
                     capacity=past + n)
    inputs = []
    for layer in range(layers):
        if past:
            k, v = _past(gen, past)
            mi.kv_cache_append(cache, layer, k, v, 0)
            del k, v
        x = _layer_inputs(case, gen)
        names = ("qp", "k", "v", "qw", "kw") if case.get("proj") else ("q", "k", "v", "gate")
        inputs.append((layer, *(x[name] for name in names)))
    engine = mi.Engine(cache, mtp_capacity=256)
    return {"case": case, "engine": engine, "cache": cache, "past": past, "inputs": inputs,
            "rows": _cache_views(cache)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ragged":
        return mi.attn_decode_ragged(state["k"], state["v"], state["offsets"], state["lengths"],
                                     state["q"], case["hi"], num_kv_heads=G, gate=state["gate"],
                                     out=state["out"], workspace=state["workspace"],
                                     validate=False)
    if kind == "oproj":
        if case["q4"]:
            return [mi.matvec_q4(x["x"], x["w"], x["scales"], x["biases"], case["group_size"])
                    for x in state["layers"]]
        return [mi.matvec_bf16(x["x"], x["w"]) for x in state["layers"]]
    engine, cache = state["engine"], state["cache"]
    cache.set_pos(state["past"])  # the pass starts where the context ends
    if kind == "token":
        out = (engine.forward_proj if case["proj"] else engine.forward)(state["inputs"])
    elif kind == "verify":
        layer, q, k, v, gate = state["inputs"][0]
        out = [mi.attn_verify(cache, layer, q, k, v, state["past"], gate=gate)]
    else:
        f = engine.forward_batched_proj if case["proj"] else engine.forward_batched
        out = f(state["inputs"])
    return {"out": out, "cache": state["rows"]}


# ------------------------------------------------------------ work, limits --


def work(case):
    kind = case["kind"]
    if kind == "oproj":
        o, i = case["out_dim"], case["in_dim"]
        w = o * i // 2 + 4 * o * (i // case["group_size"]) if case["q4"] else 2 * o * i
        return {"bytes": case["layers"] * (w + 2 * i + 4 * o), "flops": case["layers"] * 2 * o * i}
    row = 2 * 2 * KV_COLS  # K and V of one cached row
    if kind == "ragged":
        rows = case["batch"] * (case["lo"] + case["hi"]) // 2
        return {"bytes": rows * row + case["batch"] * (3 * 2 * Q_COLS + 8),
                "flops": 4 * Q_COLS * rows}
    layers, n = case.get("layers", 1), case.get("n", 1)
    past = case["pos"] if kind == "token" else case["past"]
    pairs = n * past + n * (n + 1) // 2
    # the past read once, the new rows taken and stored, queries and gates
    # taken, outputs written
    new = 4 * (2 * Q_COLS + 2 * KV_COLS) if case.get("proj") else 2 * (2 * Q_COLS + 2 * KV_COLS)
    return {"bytes": layers * (past * row + n * (new + row + 2 * Q_COLS)),
            "flops": layers * 4 * Q_COLS * pairs}


def tolerance(case):
    if case["kind"] == "oproj":
        # f32 sums of up to 8192 products: 1e-7 to 1.3e-7 from the 64-bit result
        return {"rel": 1e-6, "max": 1e-5}
    # f16 weights and outputs under f32 sums: 2.5e-4 to 5e-4 from the 64-bit
    # result
    return {"rel": 2e-3, "max": 5e-2}


# ---------------------------------------------------------- 64-bit results --


def _attend(q, k, v, gate, past):
    """q, gate [n, H, D], k, v [past + n, G, D], all f64: causal attention of
    token i over rows [0, past + i], then the sigmoid gate."""
    n = q.shape[0]
    out = torch.empty_like(q)
    rows = torch.arange(k.shape[0], device=q.device)
    per = max(1, (1 << 26) // k.shape[0])  # query rows at a time
    for h in range(H):
        kh, vh = k[:, h // (H // G)], v[:, h // (H // G)]
        for i in range(0, n, per):
            j = min(n, i + per)
            s = q[i:j, h] @ kh.t() / math.sqrt(D)
            ends = torch.arange(past + i, past + j, device=q.device)
            s.masked_fill_(rows[None, :] > ends[:, None], -math.inf)
            out[i:j, h] = torch.softmax(s, 1) @ vh
    return out * torch.sigmoid(gate)


def _norm_rope(x, w, pos):
    """RMS norm over D and NeoX rotation of the first ROTARY columns of x
    [n, heads, D] in f64; the angle of a position is an f32 product by
    definition of the operator."""
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    half = ROTARY // 2
    e = -2.0 * torch.arange(half, dtype=torch.float32) / ROTARY
    inv = torch.tensor(ROPE_THETA, dtype=torch.float32) ** e
    p = torch.arange(pos, pos + x.shape[0], dtype=torch.float32)
    a = (p[:, None] * inv[None, :]).double().to(x.device)[:, None, :]
    lo, hi = y[..., :half].clone(), y[..., half:ROTARY].clone()
    y[..., :half] = lo * a.cos() - hi * a.sin()
    y[..., half:ROTARY] = hi * a.cos() + lo * a.sin()
    return y


def _k_layout(rows):
    """[cap, G, D] rows in the device order of K: blocks of 32 rows, row w of
    a block at half (w / 4) % 2, slot 4 (w / 8) + w % 4, columns in chunks of
    eight."""
    b = rows.reshape(-1, 4, 2, 4, G, D // 8, 8)  # block, w/8, half, w%4, head, chunk, column
    return b.permute(0, 4, 2, 5, 1, 3, 6).reshape(-1)


def _v_layout(rows):
    """[cap, G, D] rows in the device order of V: transposed blocks of 8."""
    return rows.reshape(-1, 8, G, D).permute(0, 2, 3, 1).reshape(-1)


def exact(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "oproj":
        outs = []
        for _ in range(case["layers"]):
            x = _weights(case, gen)
            if case["q4"]:
                nib = torch.stack([(x["w"] >> (4 * j)) & 15 for j in range(8)], -1)
                nib = nib.reshape(case["out_dim"], -1, case["group_size"]).double()
                w = nib * x["scales"].double()[..., None] + x["biases"].double()[..., None]
                w = w.reshape(case["out_dim"], -1)
            else:
                w = x["w"].double()
            outs.append(w @ x["x"].double())
        return outs
    if kind == "ragged":
        ln, off, rows = _lengths(case, seed)
        x = _ragged_inputs(case, gen, rows)
        k, v = x["k"].view(-1, G, D), x["v"].view(-1, G, D)
        out = torch.empty(case["batch"], H, D, dtype=torch.float64, device="cuda")
        for s in range(case["batch"]):
            a, b = int(off[s]), int(off[s] + ln[s])
            out[s] = _attend(x["q"][s:s + 1].double(), k[a:b].double(), v[a:b].double(),
                             x["gate"][s:s + 1].double(), b - a - 1)[0]
        return out
    past = case["pos"] if kind == "token" else case["past"]
    n = case.get("n", 1)
    cap = max(1, -(-(past + n) // 256)) * 256
    outs, rows = [], []
    for _ in range(case.get("layers", 1)):
        k = torch.zeros(cap, G, D, dtype=torch.float64, device="cuda")
        v = torch.zeros_like(k)
        if past:
            pk, pv = _past(gen, past)
            k[:past], v[:past] = pk.view(-1, G, D).double(), pv.view(-1, G, D).double()
        x = _layer_inputs(case, gen)
        if case.get("proj"):
            qp = x["qp"].double()
            q, gate = _norm_rope(qp[..., :D], x["qw"], past), qp[..., D:]
            k[past:past + n] = _norm_rope(x["k"].double(), x["kw"], past)
            v[past:past + n] = x["v"].double()
        else:
            q, gate = x["q"].double(), x["gate"].double()
            k[past:past + n] = x["k"].view(-1, G, D).double()
            v[past:past + n] = x["v"].view(-1, G, D).double()
        o = _attend(q, k[:past + n], v[:past + n], gate, past)
        # laid out as the call returns it
        if kind == "token" and case["proj"]:
            o = o.reshape(H, D)
        outs.append(o)
        rows += [_k_layout(k), _v_layout(v)]
    return {"out": outs, "cache": rows}
