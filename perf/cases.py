"""Workloads the attention path is timed on, each through a public entry point.

A case is a dict of plain values with a ``kind``:

* ``decode``: one token per sequence over a contiguous K/V cache
  (``Qwen35RocmOps.online_attention``), uniform or ragged, optionally gated;
* ``paged_decode``: the same over a shared page pool
  (``paged_online_attention``);
* ``append_prefill``: a prompt chunk appended and attended
  (``append_prefill_attention_``);
* ``seam_prefill``: the llama batched-attention seam (``cuda.attention_batch``)
  in the engine's own float32, optionally windowed;
* ``attention_step`` / ``attention_prefill``: the Qwen3.5 attention layer for
  one token per sequence / for a prompt chunk;
* ``recurrent_step`` / ``recurrent_prefill``: the Qwen3.5 recurrent layer for
  one token per sequence / for a prompt chunk, float32 end to end;
* ``gdn_chunk``: the gated delta-rule recurrence alone over a chunk.
"""

import importlib
import math

import numpy as np
import torch

PACKAGE = "alpacca-open-sourced-by-jt_amd"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
SECTIONS = (11, 11, 10, 0)  # Qwen3.5 rotary sections: 32 pairs, 64 rotated channels
ROPE_BASE = 1.0e7
EPS = 1.0e-6
CONV_KERNEL = 4

_modules = {}


def _mod(name):
    if name not in _modules:
        _modules[name] = importlib.import_module(PACKAGE + "." + name)
    return _modules[name]


def _ops():
    if "ops" not in _modules:
        _modules["ops"] = _mod("qwen35_rocm_ops").Qwen35RocmOps(device_index=0)
    return _modules["ops"]


# ------------------------------------------------------------------ cases


def listed():
    return [
        # one chat user on a small llama in the engine's float32: the smallest
        # call, all latency
        dict(name="llama1b_decode_f32_512", kind="decode", batch=1, q_heads=32, kv_heads=8,
             dim=64, length=512, dtype="f32", ragged=False, gate=False),
        # a full serving batch at a long context: the largest read of a cache
        dict(name="llama8b_decode_f16_8k", kind="decode", batch=16, q_heads=32, kv_heads=8,
             dim=128, length=8192, dtype="f16", ragged=False, gate=False),
        # the same batch as it is in service, every sequence at its own length
        dict(name="llama8b_decode_f16_ragged", kind="decode", batch=16, q_heads=32, kv_heads=8,
             dim=128, length=8192, dtype="f16", ragged=True, gate=False),
        # serving from a page pool, sequences of ordinary lengths
        dict(name="llama8b_paged_decode_bf16_3k", kind="paged_decode", batch=8, q_heads=32,
             kv_heads=8, dim=128, length=3000, dtype="bf16", page_size=64),
        # one chunk of a long prompt
        dict(name="llama8b_prefill_bf16_2k_on_2k", kind="append_prefill", q_heads=32, kv_heads=8,
             dim=128, dtype="bf16", prefix=2048, tokens=2048),
        # the next short message of a long chat
        dict(name="llama8b_prefill_bf16_77_on_6k", kind="append_prefill", q_heads=32, kv_heads=8,
             dim=128, dtype="bf16", prefix=6011, tokens=77),
        # a prompt of the small llama through the engine's seam, float32
        dict(name="llama1b_prefill_f32_1000", kind="seam_prefill", q_heads=32, kv_heads=8,
             dim=64, prefix=0, tokens=1000, window=0),
        # Qwen3.5 attention layer, long-context decode of four users
        dict(name="qwen35_attention_step_bf16_32k", kind="attention_step", batch=4, q_heads=16,
             kv_heads=2, dim=256, length=32768, dtype="bf16"),
        # Qwen3.5 attention layer, one chunk of a long prompt
        dict(name="qwen35_attention_prefill_bf16_2k_on_2k", kind="attention_prefill", q_heads=16,
             kv_heads=2, dim=256, dtype="bf16", prefix=2048, tokens=2048),
        # Qwen3.5 recurrent layer, one decode token of one user
        dict(name="qwen35_recurrent_step_f32", kind="recurrent_step", batch=1, key_heads=16,
             value_heads=32, dim=128),
        # Qwen3.5 recurrent layer, one prompt chunk
        dict(name="qwen35_recurrent_prefill_f32_1024", kind="recurrent_prefill", tokens=1024,
             key_heads=16, value_heads=32, dim=128),
        # the recurrence alone over a bf16 chunk
        dict(name="gdn_chunk_bf16_1024", kind="gdn_chunk", batch=1, tokens=1024, key_heads=16,
             value_heads=32, dim=128, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


LLAMA_HEADS = ((32, 8), (32, 8), (24, 8), (8, 8))
QWEN_HEADS = ((16, 2), (16, 2), (8, 2), (24, 4))


def draw(rng):
    kind = rng.choice(["decode", "decode", "paged_decode", "append_prefill", "append_prefill",
                       "seam_prefill", "attention_step", "attention_prefill", "recurrent_step",
                       "recurrent_prefill", "gdn_chunk"])
    if kind in ("decode", "paged_decode"):
        q_heads, kv_heads = rng.choice(LLAMA_HEADS + QWEN_HEADS)
        dim = 256 if (q_heads, kv_heads) in QWEN_HEADS else rng.choice([64, 128, 128])
        dtype = rng.choice(["f16", "bf16", "f32"] if kind == "decode" else ["f16", "bf16"])
        if kind == "decode" and dtype != "f32" and rng.random() < 0.1:
            dim = 80
        batch = _log_int(rng, 1, 32)
        row = 2 * kv_heads * dim * BYTES[dtype] * batch
        most = min(32768, (1 << 29) // row // (8 if dim == 80 else 1))
        case = dict(kind=kind, batch=batch, q_heads=q_heads, kv_heads=kv_heads, dim=dim,
                    length=_log_int(rng, 100, most), dtype=dtype)
        if kind == "paged_decode":
            case["page_size"] = rng.choice([32, 64, 256])
        else:
            case["ragged"] = batch > 1 and rng.random() < 0.5
            case["gate"] = dim == 256 and rng.random() < 0.5
        return case
    if kind == "append_prefill":
        q_heads, kv_heads = rng.choice(LLAMA_HEADS)
        return dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, dim=rng.choice([64, 128, 128]),
                    dtype=rng.choice(["bf16", "f16"]),
                    prefix=rng.choice([0, _log_int(rng, 16, 8192)]),
                    tokens=_log_int(rng, 9, 1024))
    if kind == "seam_prefill":
        q_heads, kv_heads = rng.choice(LLAMA_HEADS)
        return dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, dim=rng.choice([64, 128]),
                    prefix=rng.choice([0, _log_int(rng, 16, 1024)]), tokens=_log_int(rng, 9, 1024),
                    window=rng.choice([0, 0, 512]))
    if kind in ("attention_step", "attention_prefill"):
        q_heads, kv_heads = rng.choice(QWEN_HEADS)
        if kind == "attention_prefill":
            return dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, dim=256,
                        dtype=rng.choice(["bf16", "f16"]),
                        prefix=rng.choice([0, _log_int(rng, 16, 8192)]),
                        tokens=_log_int(rng, 9, 1024))
        batch = _log_int(rng, 1, 16)
        row = 2 * kv_heads * 256 * 2 * batch
        return dict(kind=kind, batch=batch, q_heads=q_heads, kv_heads=kv_heads, dim=256,
                    length=_log_int(rng, 100, min(32768, (1 << 28) // row)),
                    dtype=rng.choice(["bf16", "f16"]))
    key_heads, value_heads = rng.choice([(16, 32), (16, 32), (16, 16), (8, 32)])
    if kind == "recurrent_step":
        return dict(kind=kind, batch=_log_int(rng, 1, 32), key_heads=key_heads,
                    value_heads=value_heads, dim=128)
    case = dict(kind=kind, tokens=_log_int(rng, 9, 1024), key_heads=key_heads,
                value_heads=value_heads, dim=128)
    if kind == "gdn_chunk":
        case["batch"] = _log_int(rng, 1, 4)
        case["dtype"] = rng.choice(["bf16", "bf16", "f32"])
    return case


# ------------------------------------------------------------------ inputs


class _Draw:
    """Seeded N(0, 1) and uniform tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, scale=1.0):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return (x * scale if scale != 1.0 else x).to(dtype)

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(shape, generator=self.gen, device="cuda")

    def lengths(self, lo, hi, n):
        return torch.randint(lo, hi + 1, (n,), generator=self.gen, device="cuda",
                             dtype=torch.int32)


def _ragged_lens(case, d):
    return d.lengths(max(1, case["length"] // 8), case["length"], case["batch"])


def prepare(case, seed):
    """What the caller holds before the call (see each kind's ``run``)."""
    c, d = case, _Draw(seed)
    kind = c["kind"]
    s = {"case": c}
    if kind == "decode":
        dt = DTYPES[c["dtype"]]
        s["q"] = d.normal(c["batch"], c["q_heads"], c["dim"], dtype=dt)
        for name in ("k", "v"):
            s[name] = d.normal(c["length"], c["batch"], c["kv_heads"], c["dim"], dtype=dt)
        s["lens"] = _ragged_lens(c, d) if c["ragged"] else None
        s["gate"] = d.normal(c["batch"], c["q_heads"], c["dim"], dtype=dt) if c["gate"] else None
    elif kind == "paged_decode":
        dt, ps = DTYPES[c["dtype"]], c["page_size"]
        per = (c["length"] + ps - 1) // ps
        s["q"] = d.normal(c["batch"], c["q_heads"], c["dim"], dtype=dt)
        for name in ("k", "v"):
            s[name] = d.normal(c["batch"] * per, ps, c["kv_heads"], c["dim"], dtype=dt)
        s["lens"] = _ragged_lens(c, d)
        perm = torch.randperm(c["batch"] * per, generator=d.gen, device="cuda")
        s["table"] = perm.to(torch.int32).reshape(c["batch"], per).contiguous()
    elif kind == "append_prefill":
        dt = DTYPES[c["dtype"]]
        total = c["prefix"] + c["tokens"]
        s["q"] = d.normal(c["tokens"], c["q_heads"], c["dim"], dtype=dt)
        for name in ("k", "v"):
            s[name] = d.normal(c["tokens"], c["kv_heads"], c["dim"], dtype=dt)
            cache = torch.zeros(total, 1, c["kv_heads"], c["dim"], dtype=dt, device="cuda")
            cache[:c["prefix"]] = d.normal(c["prefix"], 1, c["kv_heads"], c["dim"], dtype=dt)
            s[name + "_cache"] = cache
    elif kind == "seam_prefill":
        total = c["prefix"] + c["tokens"]
        s["q"] = d.normal(c["tokens"], c["q_heads"], c["dim"])
        s["k"] = d.normal(total, c["kv_heads"], c["dim"])
        s["v"] = d.normal(total, c["kv_heads"], c["dim"])
        s["positions"] = np.arange(c["prefix"], total)
    elif kind in ("attention_step", "attention_prefill"):
        dt, dim = DTYPES[c["dtype"]], c["dim"]
        step = kind == "attention_step"
        rows = c["batch"] if step else c["tokens"]
        batch = c["batch"] if step else 1
        total = c["length"] if step else c["prefix"] + c["tokens"]
        s["qg"] = d.normal(rows, c["q_heads"] * 2 * dim, dtype=dt)
        s["k"] = d.normal(rows, c["kv_heads"] * dim, dtype=dt)
        s["v"] = d.normal(rows, c["kv_heads"] * dim, dtype=dt)
        s["qw"] = 1.0 + d.normal(dim, scale=0.1)
        s["kw"] = 1.0 + d.normal(dim, scale=0.1)
        kept = total - 1 if step else c["prefix"]
        for name in ("k", "v"):
            cache = torch.zeros(total, batch, c["kv_heads"], dim, dtype=dt, device="cuda")
            cache[:kept] = d.normal(kept, batch, c["kv_heads"], dim, dtype=dt)
            s[name + "_cache"] = cache
    elif kind in ("recurrent_step", "recurrent_prefill"):
        hk, hv, dim = c["key_heads"], c["value_heads"], c["dim"]
        rows = c["batch"] if kind == "recurrent_step" else c["tokens"]
        channels = 2 * hk * dim + hv * dim
        s["mixed"] = d.normal(rows, channels)
        s["conv"] = d.normal(CONV_KERNEL, channels, scale=0.5)
        s["gate"] = d.normal(rows, hv * dim)
        s["beta"], s["alpha"] = d.normal(rows, hv), d.normal(rows, hv)
        s["dt"] = d.normal(hv, scale=0.5)
        s["ssm"] = -torch.exp(d.uniform(-1.0, 1.0, hv))
        s["norm"] = 1.0 + d.normal(dim, scale=0.1)
        batch = c["batch"] if kind == "recurrent_step" else 1
        ws = _ops().initialize_recurrent_workspace(
            batch_size=batch, convolution_kernel=CONV_KERNEL, convolution_channels=channels,
            value_heads=hv, value_dimension=dim, key_dimension=dim)
        ws.convolution_history.copy_(d.normal(*ws.convolution_history.shape))
        ws.delta_state.copy_(d.normal(*ws.delta_state.shape, scale=0.1))
        s["ws"] = ws
    elif kind == "gdn_chunk":
        dt, dim = DTYPES[c["dtype"]], c["dim"]
        lead = (c["batch"], c["tokens"])
        for name in ("q", "k"):
            x = d.normal(*lead, c["key_heads"], dim)
            s[name] = (x / x.norm(dim=-1, keepdim=True).clamp_min(EPS)).to(dt)
        s["v"] = d.normal(*lead, c["value_heads"], dim, dtype=dt)
        s["beta"] = torch.sigmoid(d.normal(*lead, c["value_heads"]))
        rate = torch.exp(d.uniform(-1.0, 1.0, c["value_heads"]))
        s["g"] = -rate * torch.nn.functional.softplus(d.normal(*lead, c["value_heads"]))
        s["state"] = d.normal(c["batch"], c["value_heads"], dim, dim, scale=0.1)
    else:
        raise ValueError("unknown kind " + kind)
    return s


def run(state):
    """One pass through the public entry point of the case's kind."""
    s, c = state, state["case"]
    kind, ops = c["kind"], _ops()
    if kind == "decode":
        return ops.online_attention(s["q"], s["k"], s["v"], length=c["length"],
                                    seq_lens=s["lens"], gate=s["gate"])
    if kind == "paged_decode":
        return ops.paged_online_attention(s["q"], s["k"], s["v"], s["table"],
                                          length=c["length"], seq_lens=s["lens"])
    if kind == "append_prefill":
        out, _ = ops.append_prefill_attention_(s["q"], s["k"], s["v"], s["k_cache"],
                                               s["v_cache"], position=c["prefix"])
        return out, s["k_cache"], s["v_cache"]
    if kind == "seam_prefill":
        return _mod("cuda").attention_batch(s["q"], s["k"], s["v"], s["positions"],
                                            c["q_heads"] // c["kv_heads"],
                                            1.0 / math.sqrt(c["dim"]), window=c["window"])
    if kind in ("attention_step", "attention_prefill"):
        step = kind == "attention_step"
        call = ops.attention_layer_step_ if step else ops.attention_layer_prefill_
        out, _ = call(s["qg"], s["k"], s["v"], s["qw"], s["kw"], s["k_cache"], s["v_cache"],
                      position=c["length"] - 1 if step else c["prefix"], sections=SECTIONS,
                      frequency_base=ROPE_BASE, epsilon=EPS)
        return out, s["k_cache"], s["v_cache"]
    if kind in ("recurrent_step", "recurrent_prefill"):
        call = ops.recurrent_layer_step_ if kind == "recurrent_step" else \
            ops.recurrent_layer_prefill_
        out = call(s["ws"], s["mixed"], s["conv"], s["gate"], s["beta"], s["alpha"], s["dt"],
                   s["ssm"], s["norm"], key_heads=c["key_heads"], key_dimension=c["dim"],
                   epsilon=EPS)
        return out, s["ws"].convolution_history, s["ws"].delta_state
    out = ops.gated_delta_net_chunk_(s["state"], s["q"], s["k"], s["v"], s["beta"], s["g"])
    return out, s["state"]


# ------------------------------------------------------------------ work


def _mean_ragged(case):
    return case["batch"] * (max(1, case["length"] // 8) + case["length"]) // 2


def _pairs(tokens, prefix, window):
    """Visible (query, key) pairs of a causal chunk."""
    n = tokens * prefix + tokens * (tokens + 1) // 2
    if window:
        n = sum(min(prefix + t + 1, window) for t in range(tokens))
    return n


def _gdn_flops(rows, heads, dim):
    """The token-sequential recurrence: S k, the rank-1 update, S q."""
    return 6 * rows * heads * dim * dim


def work(case):
    c, kind = case, case["kind"]
    if kind in ("decode", "paged_decode", "attention_step"):
        es = BYTES[c["dtype"]]
        ragged = kind == "paged_decode" or c.get("ragged", False)
        rows = _mean_ragged(c) if ragged else c["batch"] * c["length"]
        heads = c["batch"] * c["q_heads"] * c["dim"]
        extra = 2 * heads + (heads if kind == "attention_step" or c.get("gate") else 0)
        return {"bytes": es * (2 * rows * c["kv_heads"] * c["dim"] + extra),
                "flops": 4 * rows * c["q_heads"] * c["dim"]}
    if kind in ("append_prefill", "seam_prefill", "attention_prefill"):
        es = BYTES[c.get("dtype", "f32")]
        total = c["prefix"] + c["tokens"]
        qo = (3 if kind == "attention_prefill" else 2) * c["tokens"] * c["q_heads"] * c["dim"]
        new = 0 if kind == "seam_prefill" else 2 * c["tokens"] * c["kv_heads"] * c["dim"]
        return {"bytes": es * (qo + new + 2 * total * c["kv_heads"] * c["dim"]),
                "flops": 4 * c["dim"] * c["q_heads"] * _pairs(c["tokens"], c["prefix"],
                                                              c.get("window", 0))}
    hk, hv, dim = c["key_heads"], c["value_heads"], c["dim"]
    if kind == "gdn_chunk":
        rows, es = c["batch"] * c["tokens"], BYTES[c["dtype"]]
        io = es * rows * dim * (2 * hk + 2 * hv) + 8 * rows * hv
        return {"bytes": io + 8 * c["batch"] * hv * dim * dim, "flops": _gdn_flops(rows, hv, dim)}
    rows = c["batch"] if kind == "recurrent_step" else c["tokens"]
    seqs = c["batch"] if kind == "recurrent_step" else 1
    channels = 2 * hk * dim + hv * dim
    io = 4 * rows * (channels + 2 * hv * dim + 2 * hv) + 4 * CONV_KERNEL * channels
    held = 8 * seqs * (hv * dim * dim + (CONV_KERNEL - 1) * channels)
    return {"bytes": io + held, "flops": _gdn_flops(rows, hv, dim) + 2 * CONV_KERNEL * rows * channels}


def tolerance(case):
    """About four times the error against ``exact`` measured over the ranges:
    float32 up to 2.7e-6 (a chunk's recurrent state), float16 up to 4.2e-4,
    bfloat16 up to 3.4e-3 (probabilities, rotated rows and output rounded)
    and 1.7e-3 for the recurrence alone (output rounded once)."""
    if case["kind"] == "gdn_chunk" and case["dtype"] == "bf16":
        return {"rel": 7e-3}
    return {"rel": {"f32": 1.1e-5, "f16": 1.7e-3, "bf16": 1.3e-2}[case.get("dtype", "f32")]}


# ------------------------------------------------------------------ exact


def _attend(q, k, v, scale, first_visible=None, last_visible=None):
    """float64 softmax attention of ``q [T, Hq, D]`` over ``k, v [N, Hkv, D]``;
    query t sees rows ``first_visible[t] .. last_visible[t]``."""
    q, k, v = q.double(), k.double(), v.double()
    tokens, q_heads, _ = q.shape
    rows, kv_heads, _ = k.shape
    group = q_heads // kv_heads
    out = torch.empty_like(q)
    j = torch.arange(rows, device=q.device)
    for h in range(kv_heads):
        kh, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for t0 in range(0, tokens, 512):
            t1 = min(tokens, t0 + 512)
            qs = q[t0:t1, h * group:(h + 1) * group].reshape(-1, q.shape[2])
            score = (qs @ kh) * scale
            if last_visible is not None:
                hide = j[None, :] > last_visible[t0:t1, None]
                if first_visible is not None:
                    hide = hide | (j[None, :] < first_visible[t0:t1, None])
                score = score.masked_fill(hide.repeat_interleave(group, 0), -math.inf)
            p = torch.softmax(score, dim=-1)
            out[t0:t1, h * group:(h + 1) * group] = (p @ vh).reshape(t1 - t0, group, -1)
    return out


def _rms(x, weight):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * weight.double()


def _rope(x, positions):
    """Half-split rotation of the first 64 channels of ``x [T, H, D]``."""
    pairs = sum(SECTIONS)
    inv = ROPE_BASE ** (-2.0 * torch.arange(pairs, device=x.device).double() / (2 * pairs))
    angle = (positions.double()[:, None] * inv)[:, None, :]
    a, b = x[..., :pairs], x[..., pairs:2 * pairs]
    turned = [a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()]
    return torch.cat(turned + [x[..., 2 * pairs:]], dim=-1)


def _gdn(state, q, k, v, beta, g):
    """float64 token-by-token recurrence: ``state [Hv, Dv, Dk]`` in place."""
    hv, hk = v.shape[1], q.shape[1]
    rep = hv // hk
    q, k = q.double().repeat(1, rep, 1), k.double().repeat(1, rep, 1)
    v, beta, decay = v.double(), beta.double(), torch.exp(g.double())
    out = torch.empty_like(v)
    for t in range(v.shape[0]):
        state.mul_(decay[t][:, None, None])
        pred = (state * k[t][:, None, :]).sum(-1)
        state.add_((beta[t][:, None] * (v[t] - pred))[:, :, None] * k[t][:, None, :])
        out[t] = (state * q[t][:, None, :]).sum(-1)
    return out / math.sqrt(q.shape[2])


def _recurrent(s, hk, hv, dim, mixed, gate, beta, alpha, history, state):
    """float64 recurrent layer over the tokens of one sequence."""
    window = torch.cat([history.double(), mixed.double()])
    tokens = mixed.shape[0]
    conv = sum(window[i:i + tokens] * s["conv"][i].double() for i in range(CONV_KERNEL))
    conv = conv * torch.sigmoid(conv)
    q, k, v = conv.split([hk * dim, hk * dim, hv * dim], dim=1)

    def unit(x):
        x = x.reshape(tokens, hk, dim)
        return x / x.norm(dim=-1, keepdim=True).clamp_min(EPS)

    step = torch.nn.functional.softplus(alpha.double() + s["dt"].double())
    out = _gdn(state, unit(q), unit(k), v.reshape(tokens, hv, dim), torch.sigmoid(beta.double()),
               step * s["ssm"].double())
    z = gate.double().reshape(tokens, hv, dim)
    out = _rms(out, s["norm"]) * z * torch.sigmoid(z)
    return out.reshape(tokens, hv * dim), window[-(CONV_KERNEL - 1):]


def exact(case, seed):
    """``run``'s outputs for these inputs in float64."""
    c, s = case, prepare(case, seed)
    kind = c["kind"]
    scale = 1.0 / math.sqrt(c["dim"])
    if kind in ("decode", "paged_decode"):
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for b in range(c["batch"]):
            n = c["length"] if s["lens"] is None else int(s["lens"][b])
            if kind == "decode":
                k, v = s["k"][:n, b], s["v"][:n, b]
            else:
                pages = s["table"][b].long()
                k, v = (x[pages].flatten(0, 1)[:n] for x in (s["k"], s["v"]))
            out[b] = _attend(s["q"][b:b + 1], k, v, scale)[0]
        if s.get("gate") is not None:
            out = out * torch.sigmoid(s["gate"].double())
        return out
    if kind == "append_prefill":
        k, v = s["k_cache"].clone(), s["v_cache"].clone()
        k[c["prefix"]:, 0], v[c["prefix"]:, 0] = s["k"], s["v"]
        last = torch.arange(c["prefix"], c["prefix"] + c["tokens"], device="cuda")
        return _attend(s["q"], k[:, 0], v[:, 0], scale, None, last), k, v
    if kind == "seam_prefill":
        last = torch.arange(c["prefix"], c["prefix"] + c["tokens"], device="cuda")
        first = last - c["window"] + 1 if c["window"] else None
        return _attend(s["q"], s["k"], s["v"], scale, first, last).flatten(1)
    if kind in ("attention_step", "attention_prefill"):
        step = kind == "attention_step"
        dim, rows = c["dim"], s["qg"].shape[0]
        at = c["length"] - 1 if step else c["prefix"]
        pos = torch.full((rows,), at, device="cuda") if step else \
            torch.arange(at, at + rows, device="cuda")
        q, z = s["qg"].double().reshape(rows, c["q_heads"], 2 * dim).split(dim, dim=-1)
        q = _rope(_rms(q, s["qw"]), pos)
        new_k = _rope(_rms(s["k"].reshape(rows, c["kv_heads"], dim), s["kw"]), pos)
        new_v = s["v"].reshape(rows, c["kv_heads"], dim)
        k, v = s["k_cache"].double(), s["v_cache"].double()
        if step:
            k[at], v[at] = new_k, new_v.double()
            out = torch.stack([_attend(q[b:b + 1], k[:, b], v[:, b], scale)[0]
                               for b in range(rows)])
        else:
            k[at:, 0], v[at:, 0] = new_k, new_v.double()
            out = _attend(q, k[:, 0], v[:, 0], scale, None, pos)
        return out * torch.sigmoid(z), k, v
    if kind in ("recurrent_step", "recurrent_prefill"):
        hk, hv, dim = c["key_heads"], c["value_heads"], c["dim"]
        history, state = s["ws"].convolution_history.double(), s["ws"].delta_state.double()
        outs = []
        for b in range(state.shape[0]):
            rows = slice(b, b + 1) if kind == "recurrent_step" else slice(None)
            o, history[b] = _recurrent(s, hk, hv, dim, s["mixed"][rows], s["gate"][rows],
                                       s["beta"][rows], s["alpha"][rows], history[b], state[b])
            outs.append(o)
        return torch.cat(outs), history, state
    state = s["state"].double()
    outs = [_gdn(state[b], s["q"][b], s["k"][b], s["v"][b], s["beta"][b], s["g"][b])
            for b in range(c["batch"])]
    return torch.stack(outs), state
