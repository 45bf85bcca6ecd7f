"""Timed cases of the hybrid-backbone prefill path: what a program that serves
or checks the backbone calls, through the Python binding of the C ABI.

Kinds of case (sizes in tokens; widths are the layer shapes of
workloads.block_config: hidden 2048, MLP 6144, DeltaNet 16/32 heads x 128,
attention 16 q / 2 kv heads x 256):

  prefill    one whole request: ids in, final hidden states and pooled logits out,
             alone or resumed from a cached prefix
  gemm       one projection y = x w^T
  mlp        one MLP block on the residual stream: norm, SwiGLU, down-projection
  scan       one gated-DeltaNet scan, alone, resumed, captured, or a ragged batch
  attention  one gated attention core: q/k norm + rotary, value layout, attention
  mixer      what stands around the scan in a DeltaNet layer: conv, gates, gated norm
"""
import importlib
import math
import random

import numpy as np
import torch

clef = importlib.import_module("clef-rs_amd.clef_hip")
workloads = importlib.import_module("clef-rs_amd.workloads")

DEV = "cuda"
CFG = workloads.block_config()
HID, MID = CFG["hidden_size"], CFG["intermediate_size"]
HK, HV, DH = CFG["linear_num_key_heads"], CFG["linear_num_value_heads"], CFG["linear_key_head_dim"]
HEADS, KVH, AD = CFG["num_attention_heads"], CFG["num_key_value_heads"], CFG["head_dim"]
TAPS = CFG["linear_conv_kernel_dim"]
THETA = CFG["rope_parameters"]["rope_theta"]
ROT = int(AD * CFG["rope_parameters"]["partial_rotary_factor"])
EPS = CFG["rms_norm_eps"]
KEY, VALUE = HK * DH, HV * DH
WIDTH = 2 * KEY + VALUE          # conv channels [q | k | v]
PROJ = WIDTH + VALUE             # DeltaNet in-projection columns [q | k | v | z]
ATT = 2 * HEADS * AD + 2 * KVH * AD  # attention in-projection columns [q, gate | k | v]
DT = {"f16": torch.float16, "f32": torch.float32}

# (N, K) of the projections: DeltaNet and attention in-projections, output
# projection, MLP down-projection, and the 2048-wide sweep of the benchmark
PROJECTIONS = [(PROJ, HID), (ATT, HID), (HID, VALUE), (HID, MID), (8192, 2048), (2048, 2048)]


def listed():
    return [
        # a long prompt through the block: the benchmark's step
        {"name": "prefill_4096", "kind": "prefill", "profile": "mixed", "tokens": 4096, "prefix": 0},
        # a short question behind a cached prompt: what a prefix hit serves
        {"name": "resume_100", "kind": "prefill", "profile": "mixed", "tokens": 100, "prefix": 512},
        # the widest projection of a long prompt
        {"name": "gemm_f16_in_4096", "kind": "gemm", "dtype": "f16", "m": 4096, "n": PROJ, "k": HID},
        # the MLP of a very short request, where the weights' bytes and the launches count
        {"name": "mlp_f16_33", "kind": "mlp", "dtype": "f16", "m": 33},
        # the MLP of a mid-sized request that is no multiple of any tile
        {"name": "mlp_f16_1000", "kind": "mlp", "dtype": "f16", "m": 1000},
        # a projection of the f32 profile (the parity and evaluation profile)
        {"name": "gemm_f32_2048", "kind": "gemm", "dtype": "f32", "m": 2048, "n": 8192, "k": 2048},
        # the DeltaNet scan of a long prompt
        {"name": "scan_mixed_4096", "kind": "scan", "precision": "mixed", "tokens": 4096, "requests": 1,
         "initial": False, "capture": 0},
        # the f32 scan of a resumed request
        {"name": "scan_strict_1000", "kind": "scan", "precision": "strict", "tokens": 1000, "requests": 1,
         "initial": True, "capture": 0},
        # a batch of uneven requests behind one shared prefix state
        {"name": "scan_ragged_8", "kind": "scan", "precision": "mixed", "tokens": 5003, "requests": 8,
         "initial": True, "capture": 0},
        # the attention core of a long prompt
        {"name": "attention_f16_4096", "kind": "attention", "dtype": "f16", "tokens": 4096, "prefix": 0},
        # the attention core of the f32 profile behind a cached prefix
        {"name": "attention_f32_777", "kind": "attention", "dtype": "f32", "tokens": 777, "prefix": 256},
        # the memory-bound passes around the scan
        {"name": "mixer_f16_4096", "kind": "mixer", "dtype": "f16", "tokens": 4096, "history": 0},
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of lo..hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prefill", "gemm", "gemm", "mlp", "scan", "scan", "attention", "attention", "mixer"])
    if kind == "prefill":
        profile = rng.choice(["mixed", "mixed", "mixed", "f32"])
        prefix = rng.choice([0, 0, 256, 512, 8 * rng.randint(1, 64)])
        hi = 4096 - prefix if profile == "mixed" else 512
        return {"kind": kind, "profile": profile, "tokens": _log(rng, 8, hi), "prefix": prefix}
    if kind == "gemm":
        n, k = rng.choice(PROJECTIONS + [(8 * rng.randint(8, 640), 64 * rng.randint(1, 64))])
        dtype = rng.choice(["f16", "f16", "f32"])
        return {"kind": kind, "dtype": dtype, "m": _log(rng, 1, 4096 if dtype == "f16" else 2048), "n": n, "k": k}
    if kind == "mlp":
        dtype = rng.choice(["f16", "f16", "f32"])
        return {"kind": kind, "dtype": dtype, "m": _log(rng, 1, 4096 if dtype == "f16" else 1024)}
    if kind == "scan":
        t = _log(rng, 16, 4096)
        requests = rng.choice([1, 1, rng.randint(2, 16)])
        capture = rng.randint(1, t) if requests == 1 and rng.random() < 0.3 else 0
        return {"kind": kind, "precision": rng.choice(["mixed", "mixed", "strict"]), "tokens": t,
                "requests": min(requests, t), "initial": rng.random() < 0.5, "capture": capture}
    if kind == "attention":
        dtype = rng.choice(["f16", "f16", "f32"])
        prefix = rng.choice([0, 0, 256, 512, rng.randint(1, 1000)])
        return {"kind": kind, "dtype": dtype, "tokens": _log(rng, 8, 4096 - prefix if dtype == "f16" else 1024),
                "prefix": prefix}
    return {"kind": kind, "dtype": rng.choice(["f16", "f16", "f32"]), "tokens": _log(rng, 8, 4096),
            "history": rng.choice([0, TAPS - 1])}


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device=DEV) * std).to(dtype)


def _decay(g):
    """dt bias and A_log per head: per-token decay rates from slow to fast heads."""
    rate = torch.exp(torch.empty(HV, device=DEV).uniform_(math.log(0.02), math.log(4.0), generator=g))
    return _randn(g, HV, std=0.5), torch.log(rate)


def _offsets(case):
    """Token offsets of a scan's requests: uneven lengths fixed by the case."""
    t, n = case["tokens"], case["requests"]
    cuts = sorted(random.Random(t * 4099 + n).sample(range(1, t), n - 1))
    return [0] + cuts + [t]


def _weights(seed, dtype):
    g = _gen(seed)
    out = {}
    for name, shape in workloads.weight_shapes(CFG):
        leaf = name.rsplit(".", 2)[-2:]
        if leaf[-1] in ("dt_bias", "A_log"):
            dt, a_log = _decay(g)
            out[name] = dt if leaf[-1] == "dt_bias" else a_log
        elif "conv1d" in leaf:
            out[name] = _randn(g, *shape, std=0.3)
        elif len(shape) == 1:  # norm weights; the gated norm's has no (1 + w) offset
            out[name] = _randn(g, *shape, std=0.1) + (1.0 if ".linear_attn.norm" in name else 0.0)
        else:
            out[name] = torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, 0.02, generator=g)
    return out


def _ids(case, seed):
    return np.random.default_rng(seed).integers(0, CFG["vocab_size"], case["prefix"] + case["tokens"])


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind == "prefill":
        dt = DT["f16" if case["profile"] == "mixed" else "f32"]
        model = clef.Backbone(CFG, _weights(seed, dt), profile=case["profile"], max_tokens=4096)
        ids, p = _ids(case, seed), case["prefix"]
        initial = model.prefill(ids[:p + 1], capture=p)[1] if p else None
        return {"kind": kind, "model": model, "ids": ids[p:], "initial": initial,
                "head": _randn(_gen(seed + 1), 3, HID, std=0.02)}
    if kind == "gemm":
        dt = DT[case["dtype"]]
        return {"kind": kind, "x": _randn(g, case["m"], case["k"], dtype=dt),
                "w": _randn(g, case["n"], case["k"], std=0.02, dtype=dt)}
    if kind == "mlp":
        dt = DT[case["dtype"]]
        return {"kind": kind, "dtype": dt, "h": _randn(g, case["m"], HID), "norm": 1.0 + _randn(g, HID, std=0.1),
                "gate": _randn(g, MID, HID, std=0.02, dtype=dt), "up": _randn(g, MID, HID, std=0.02, dtype=dt),
                "down": _randn(g, HID, MID, std=0.02, dtype=dt)}
    if kind == "scan":
        t = case["tokens"]
        dt = torch.float16 if case["precision"] == "mixed" else torch.float32
        mixed = torch.nn.functional.silu(_randn(g, t, WIDTH)).to(dt)  # what the conv leaves: [q | k | v]
        bias, a_log = _decay(g)
        decay = -torch.exp(a_log) * torch.nn.functional.softplus(_randn(g, t, HV) + bias)
        s = {"kind": kind, "scan": clef.DeltaScan(DH, DH, case["precision"]), "mixed": mixed, "g": decay,
             "beta": torch.sigmoid(_randn(g, t, HV)), "initial": None, "cu": None, "capture": case["capture"]}
        if case["initial"]:
            s["initial"] = _randn(g, HV, DH, DH, std=0.1)
        if case["requests"] > 1:
            s["cu"] = torch.tensor(_offsets(case), dtype=torch.int32, device=DEV)
        return s
    if kind == "attention":
        dt, t, p = DT[case["dtype"]], case["tokens"], case["prefix"]
        kn = p + t
        s = {"kind": kind, "dtype": dt, "proj": _randn(g, t, ATT, dtype=dt), "prefix": p,
             "q_norm": 1.0 + _randn(g, AD, std=0.1), "k_norm": 1.0 + _randn(g, AD, std=0.1),
             "k": torch.zeros((KVH, kn, AD), dtype=dt, device=DEV),
             "vt": torch.zeros((KVH, AD, (kn + 63) // 64 * 64), dtype=dt, device=DEV)}
        s["k"][:, :p] = _randn(g, KVH, p, AD, dtype=dt)
        s["vt"][:, :, :p] = _randn(g, KVH, AD, p, dtype=dt)
        return s
    dt, t = DT[case["dtype"]], case["tokens"]
    bias, a_log = _decay(g)
    w_ab = _randn(g, 2 * HV, HID, std=0.02, dtype=dt)
    return {"kind": kind, "dtype": dt, "h": _randn(g, t, HID), "norm": 1.0 + _randn(g, HID, std=0.1),
            "proj": _randn(g, t, PROJ, dtype=dt), "o": _randn(g, t, HV, DH, std=0.1, dtype=dt),
            "conv": _randn(g, WIDTH, TAPS, std=0.3), "dt_bias": bias, "a_log": a_log,
            "gated": 1.0 + _randn(g, DH, std=0.1), "w_ab": w_ab,
            "packed": clef.delta_gates_pack(w_ab) if dt == torch.float16 else None,
            "history": _randn(g, case["history"], WIDTH) if case["history"] else None}


# --------------------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "prefill":
        hidden, _ = s["model"].prefill(s["ids"], initial=s["initial"])
        return {"hidden": hidden, "logits": clef.head_logits(hidden[-1], s["head"])}
    if kind == "gemm":
        return clef.gemm(s["x"], s["w"])
    if kind == "mlp":
        h = s["h"].clone()  # the block's input stays with the caller
        x = clef.rms_norm(h, s["norm"], EPS, out_dtype=s["dtype"])
        return clef.gemm(clef.gemm_swiglu(x, s["gate"], s["up"]), s["down"], residual=h)
    if kind == "scan":
        q, k, v = _qkv(s["mixed"])
        if s["cu"] is not None:
            return s["scan"].prefill_varlen(q, k, v, s["g"], s["beta"], s["cu"], initial=s["initial"],
                                            out_dtype=s["mixed"].dtype)
        return s["scan"].prefill(q, k, v, s["g"], s["beta"], initial=s["initial"], capture=s["capture"],
                                 out_dtype=s["mixed"].dtype)
    if kind == "attention":
        p, dt = s["prefix"], s["dtype"]
        q, gate, k, v = _attention_views(s["proj"])
        clef.qk_norm_rotary(k, KVH, AD, s["k_norm"], ROT, THETA, pos0=p, out=s["k"], dst_offset=p)
        clef.values_transposed(v, KVH, AD, out=s["vt"], dst_offset=p)
        if dt == torch.float16:
            table = clef.rotary_table(q.shape[0], ROT, THETA, pos0=p)
            y = clef.attention_gated_qnorm(q, HEADS, s["q_norm"], EPS, table, s["k"], s["vt"], gate, 2 * AD)
        else:
            qh = clef.qk_norm_rotary(q, HEADS, AD, s["q_norm"], ROT, THETA, pos0=p, head_stride=2 * AD)
            y = clef.attention_gated(qh, s["k"], s["vt"], gate)
        return {"y": y, "k": s["k"], "vt": s["vt"]}
    dt, proj = s["dtype"], s["proj"]
    x = clef.rms_norm(s["h"], s["norm"], EPS, out_dtype=dt)
    mixed = clef.conv_silu(proj[:, :WIDTH], s["conv"], s["history"], out_dtype=dt)
    if s["packed"] is not None:
        g, beta = clef.delta_gates_proj(x, s["packed"], HV, s["dt_bias"], s["a_log"])
    else:
        ab = clef.gemm(x, s["w_ab"])
        g, beta = clef.delta_gates(ab[:, :HV], ab[:, HV:], s["dt_bias"], s["a_log"])
    y = clef.gated_rms_silu(s["o"], proj[:, WIDTH:], s["gated"], EPS, out_dtype=dt)
    return {"x": x, "mixed": mixed, "g": g, "beta": beta, "y": y}


def _qkv(m):
    t = m.shape[0]
    return (m[:, :KEY].view(t, HK, DH), m[:, KEY:2 * KEY].view(t, HK, DH), m[:, 2 * KEY:].view(t, HV, DH))


def _attention_views(proj):
    t, n = proj.shape[0], 2 * HEADS * AD
    gate = proj[:, :n].view(t, HEADS, 2 * AD)[:, :, AD:]
    return proj[:, :n], gate, proj[:, n:n + KVH * AD], proj[:, n + KVH * AD:]


# --------------------------------------------------------------------------- least work
def work(case):
    kind = case["kind"]
    if kind == "prefill":
        t, p = case["tokens"], case["prefix"]
        e = 2 if case["profile"] == "mixed" else 4
        per_token = workloads.block_flops_per_token(CFG, 0)
        per_token -= 2 * HEADS * AD  # attention pairs are counted below
        pairs = t * p + t * (t + 1) / 2
        weights = sum(math.prod(sh) for n, sh in workloads.weight_shapes(CFG) if "embed" not in n)
        cached = p * (4 * HID + 2 * e * KVH * AD) + (3 * 4 * HV * DH * DH if p else 0)
        return {"bytes": e * (weights + t * HID) + 4 * (t + p) * HID + cached,
                "flops": t * per_token + 4 * HEADS * AD * pairs + 3 * t * 6 * HV * DH * DH}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (2 if case["dtype"] == "f16" else 4) * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, e = case["m"], 2 if case["dtype"] == "f16" else 4
        return {"bytes": 3 * e * HID * MID + 8 * m * HID, "flops": 6 * m * HID * MID}
    if kind == "scan":
        t, e = case["tokens"], 2 if case["precision"] == "mixed" else 4
        states = case["requests"] + (1 if case["initial"] else 0) + (1 if case["capture"] else 0)
        return {"bytes": e * t * (WIDTH + VALUE) + 8 * t * HV + 4 * states * HV * DH * DH,
                "flops": 6 * t * HV * DH * DH}
    if kind == "attention":
        t, p, e = case["tokens"], case["prefix"], 2 if case["dtype"] == "f16" else 4
        return {"bytes": e * (t * ATT + t * HEADS * AD + 2 * KVH * AD * (2 * t + p)),
                "flops": 4 * HEADS * AD * (t * p + t * (t + 1) / 2)}
    t, e = case["tokens"], 2 if case["dtype"] == "f16" else 4
    return {"bytes": t * HID * (4 + e) + e * t * (PROJ + WIDTH + 2 * VALUE) + 8 * t * HV + e * 2 * HV * HID,
            "flops": 2 * t * 2 * HV * HID}


# --------------------------------------------------------------------------- tolerances
def tolerance(case):
    """About four times the distance from the 64-bit result that the path shows."""
    kind = case["kind"]
    half = case.get("dtype") == "f16" or case.get("profile") == "mixed" or case.get("precision") == "mixed"
    if kind == "prefill":
        return {"rel": 2e-2} if half else {"rel": 2e-5}
    if kind == "attention":  # f32: the rounding of the rotary angles
        return {"rel": 2e-3} if half else {"rel": 1.5e-5}
    if kind == "scan":
        return {"rel": 1.6e-3} if half else {"rel": 5e-6}
    return {"rel": 1.5e-3} if half else {"rel": 2e-6}


# --------------------------------------------------------------------------- 64-bit results
def _rms64(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _silu64(x):
    return x * torch.sigmoid(x)


def _conv64(x, w, history):
    """Causal conv of x [T, W] with taps oldest to newest, then SiLU."""
    t = x.shape[0]
    pad = torch.zeros((TAPS - 1, x.shape[1]), dtype=torch.float64, device=DEV)
    if history is not None:
        pad[TAPS - 1 - history.shape[0]:] = history.double()
    x = torch.cat([pad, x])
    return _silu64(sum(x[i:i + t] * w[:, i] for i in range(TAPS)))


def _scan64(q, k, v, g, beta, state, capture=0):
    """The recurrence token by token; returns o [T, HV, DH], the state after `capture`, the last state."""
    q, k, v, g, beta = (x.double() for x in (q, k, v, g, beta))
    q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + 1e-6) / math.sqrt(DH)
    k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    q, k = (x.repeat_interleave(HV // HK, 1).unsqueeze(-1) for x in (q, k))
    decay = g.exp()[:, :, None, None]
    s = torch.zeros((HV, DH, DH), dtype=torch.float64, device=DEV) if state is None else state.double()
    out, kept = torch.empty_like(v), None
    for t in range(v.shape[0]):
        s = s * decay[t]
        d = (v[t] - (s * k[t]).sum(1)) * beta[t][:, None]
        s = s + k[t] * d.unsqueeze(1)
        out[t] = (s * q[t]).sum(1)
        if t + 1 == capture:
            kept = s
    return out, kept, s


def _rotary64(x, pos0):
    """Rotate-half on the first ROT features of x [T, heads, AD]."""
    t, h = x.shape[0], ROT // 2
    freq = THETA ** (-torch.arange(h, dtype=torch.float64, device=DEV) * 2 / ROT)
    a = (pos0 + torch.arange(t, dtype=torch.float64, device=DEV))[:, None, None] * freq
    u, w = x[..., :h], x[..., h:ROT]
    return torch.cat([u * a.cos() - w * a.sin(), w * a.cos() + u * a.sin(), x[..., ROT:]], -1)


def _attention64(q, k, v, gate):
    """q, gate [T, HEADS, AD]; k, v [KN, KVH, AD]; causal, bottom-right aligned."""
    t, kn = q.shape[0], k.shape[0]
    hidden = torch.ones((t, kn), dtype=torch.bool, device=DEV).triu(kn - t + 1)
    y = torch.empty_like(q)
    for h in range(HEADS):
        kv = h // (HEADS // KVH)
        scores = (q[:, h] @ k[:, kv].t() / math.sqrt(AD)).masked_fill(hidden, -math.inf)
        y[:, h] = torch.softmax(scores, -1) @ v[:, kv]
    return (y * torch.sigmoid(gate)).reshape(t, HEADS * AD)


def _gates64(a, b, bias, a_log):
    return torch.nn.functional.softplus(a + bias) * -a_log.exp(), torch.sigmoid(b)


def _prefill64(w, ids):
    P = "model.language_model."
    get = lambda n: w[P + n].double()  # noqa: E731
    ids = torch.as_tensor(ids, device=DEV)
    h = w[P + "embed_tokens.weight"][ids].double()
    t = h.shape[0]
    for i, kind in enumerate(CFG["layer_types"]):
        p = f"layers.{i}."
        x = _rms64(h, 1.0 + get(p + "input_layernorm.weight"))
        if kind == "full_attention":
            a = p + "self_attn."
            qg = (x @ get(a + "q_proj.weight").t()).view(t, HEADS, 2 * AD)
            k, v = ((x @ get(a + n).t()).view(t, KVH, AD) for n in ("k_proj.weight", "v_proj.weight"))
            q = _rotary64(_rms64(qg[:, :, :AD], 1.0 + get(a + "q_norm.weight")), 0)
            k = _rotary64(_rms64(k, 1.0 + get(a + "k_norm.weight")), 0)
            h = h + _attention64(q, k, v, qg[:, :, AD:]) @ get(a + "o_proj.weight").t()
        else:
            a = p + "linear_attn."
            mixed = _conv64(x @ get(a + "in_proj_qkv.weight").t(), get(a + "conv1d.weight")[:, 0], None)
            g, beta = _gates64(x @ get(a + "in_proj_a.weight").t(), x @ get(a + "in_proj_b.weight").t(),
                               get(a + "dt_bias"), get(a + "A_log"))
            o = _rms64(_scan64(*_qkv(mixed), g, beta, None)[0], get(a + "norm.weight"))
            z = (x @ get(a + "in_proj_z.weight").t()).view(t, HV, DH)
            h = h + (o * _silu64(z)).reshape(t, VALUE) @ get(a + "out_proj.weight").t()
        x = _rms64(h, 1.0 + get(p + "post_attention_layernorm.weight"))
        m = _silu64(x @ get(p + "mlp.gate_proj.weight").t()) * (x @ get(p + "mlp.up_proj.weight").t())
        h = h + m @ get(p + "mlp.down_proj.weight").t()
    return _rms64(h, 1.0 + get("norm.weight"))


def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill":
        dt = DT["f16" if case["profile"] == "mixed" else "f32"]
        hidden = _prefill64(_weights(seed, dt), _ids(case, seed))
        return {"hidden": hidden, "logits": _randn(_gen(seed + 1), 3, HID, std=0.02).double() @ hidden[-1]}
    s = prepare(case, seed)
    if kind == "gemm":
        return s["x"].double() @ s["w"].double().t()
    if kind == "mlp":
        x = _rms64(s["h"].double(), s["norm"].double())
        gate, up, down = (s[n].double().t() for n in ("gate", "up", "down"))
        return s["h"].double() + (_silu64(x @ gate) * (x @ up)) @ down
    if kind == "scan":
        q, k, v = _qkv(s["mixed"])
        if s["cu"] is None:
            return _scan64(q, k, v, s["g"], s["beta"], s["initial"], s["capture"])
        parts = [_scan64(*(x[a:b] for x in (q, k, v, s["g"], s["beta"])), s["initial"])
                 for a, b in zip(_offsets(case), _offsets(case)[1:])]
        return torch.cat([o for o, _, _ in parts]), torch.stack([f for _, _, f in parts])
    if kind == "attention":
        t, p = case["tokens"], case["prefix"]
        q, gate, k, v = (x.double() for x in _attention_views(s["proj"]))
        q = _rotary64(_rms64(q.reshape(t, HEADS, 2 * AD)[:, :, :AD], s["q_norm"].double()), p)
        kc, vt = s["k"].double(), s["vt"].double()
        kc[:, p:] = _rotary64(_rms64(k.reshape(t, KVH, AD), s["k_norm"].double()), p).transpose(0, 1)
        vt[:, :, p:p + t] = v.reshape(t, KVH, AD).permute(1, 2, 0)
        y = _attention64(q, kc.transpose(0, 1), vt[:, :, :p + t].permute(2, 0, 1), gate)
        return {"y": y, "k": kc, "vt": vt}
    t, proj = case["tokens"], s["proj"].double()
    x = _rms64(s["h"].double(), s["norm"].double())
    a, b = (x @ w.double().t() for w in (s["w_ab"][:HV], s["w_ab"][HV:]))
    g, beta = _gates64(a, b, s["dt_bias"].double(), s["a_log"].double())
    y = _rms64(s["o"].double(), s["gated"].double()) * _silu64(proj[:, WIDTH:].reshape(t, HV, DH))
    return {"x": x, "mixed": _conv64(proj[:, :WIDTH], s["conv"].double(), s["history"]), "g": g, "beta": beta,
            "y": y.reshape(t, VALUE)}
