"""The workloads this library's speed is judged on.

Each case is a call, or the few calls in a row, that a program serving GGUF
models makes through `cretif_amd`: one token's matrix products, a decode
batch's FFN block, a prompt's products and its attention, the attention of one
token over a long cache, a captured decode step, and a prompt through the whole
step.  `listed()` holds the named ones, `draw()` gives others of the same
ranges, `exact()` the same results in float64 from plain torch.
"""
from __future__ import annotations

import math

import torch

import cretif_amd as cri

BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q5_0": (32, 22), "q4_k": (256, 144), "q6_k": (256, 210),
         "fp16": (1, 2)}
EPS = 1e-5
THETA = 500000.0


# --------------------------------------------------------------------------- cases

# the 16-layer 1B-parameter shape of the benchmark's decode step
ONE_B = {"layers": 16, "dim": 2048, "heads": 32, "kv_heads": 8, "head_dim": 64, "ffn": 8192, "vocab": 128256,
         "fmt": "q4_k", "head": "q6_k", "table": "q8_0"}


def listed():
    return [
        # the smallest product in use: a 135M model's FFN gate for one token; latency and the launch
        {"name": "gemv_small", "kind": "matmul", "fmt": "q8_0", "M": 1, "N": 1536, "K": 576, "ws": False},
        # one token's gate (or up) projection of a 1B model, the benchmark's headline
        {"name": "gemv_gate", "kind": "matmul", "fmt": "q4_k", "M": 1, "N": 8192, "K": 2048, "ws": False},
        # one token's LM head over a 128k vocabulary: the longest single product of decoding
        {"name": "lm_head", "kind": "matmul", "fmt": "q6_k", "M": 1, "N": 128256, "K": 2048, "ws": False},
        # the FFN block of a decode batch of 16 sequences (two fused calls)
        {"name": "ffn_batch16", "kind": "ffn", "fmt": "q4_k", "M": 16, "dim": 2048, "ffn": 8192},
        # a 512-token prompt's gate projection
        {"name": "prefill_gate_512", "kind": "matmul", "fmt": "q4_k", "M": 512, "N": 8192, "K": 2048, "ws": False},
        # a 2048-token prompt's down projection, the caller keeping a workspace
        {"name": "prefill_down_2048", "kind": "matmul", "fmt": "q8_0", "M": 2048, "N": 2048, "K": 8192, "ws": True},
        # the fused q/k/v projection of a prompt of no particular length
        {"name": "prefill_qkv_777", "kind": "matmul", "fmt": "q6_k", "M": 777, "N": 3072, "K": 2048, "ws": False},
        # the attention of a 2048-token prompt, queries read from the fused q/k/v buffer
        {"name": "attention_prompt", "kind": "prompt_attention", "heads": 32, "kv_heads": 8, "head_dim": 64,
         "M": 2048, "pos": 0},
        # the attention of one token late in a long conversation
        {"name": "attention_token", "kind": "token_attention", "heads": 32, "kv_heads": 8, "head_dim": 64, "T": 8191},
        # one decoded token of a 1B model as a serving loop replays it
        dict(ONE_B, name="step_1", kind="step", M=1, pos=2047, max_seq=2048),
        # one decode step of a batch of 16
        dict(ONE_B, name="step_16", kind="step", M=16, pos=2032, max_seq=2048),
        # a 512-token prompt through every layer, the last token's logits
        dict(ONE_B, name="prompt_512", kind="prompt", M=512, pos=0, max_seq=2048),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_k(rng, fmt, hi=8192):
    """A row length: the models' own widths and others of the block size."""
    if BLOCK[fmt][0] == 32 and rng.random() < 0.2:
        return rng.choice([576, 960, 1536 + 32, 2880])
    if rng.random() < 0.5:
        return rng.choice([k for k in (1024, 1536, 2048, 3072, 4096, 8192) if k <= hi])
    return 256 * _log_int(rng, 1, hi // 256)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "batch", "prefill", "prefill", "prefill", "ffn", "prompt_attention",
                       "prompt_attention", "token_attention", "step", "prompt"])
    fmt = rng.choice(["q4_k", "q8_0", "q6_k", "q4_0", "q5_0", "fp16", "q4_k", "q6_k"])
    if kind in ("gemv", "batch"):
        m = 1 if kind == "gemv" else rng.randint(2, 16)
        k = _draw_k(rng, fmt)
        n = _log_int(rng, 256, 128256 if k <= 4096 else 32768)
        ws = rng.random() < 0.3
        return {"kind": "matmul", "fmt": fmt, "M": m, "N": n - n % 4 if ws else n, "K": k, "ws": ws}
    if kind == "prefill":
        m, k = _log_int(rng, 17, 2048), _draw_k(rng, fmt)
        n = min(_log_int(rng, 256, 16384), (2048 * 2048 * 8192) // (m * k))
        ws = rng.random() < 0.4
        return {"kind": "matmul", "fmt": fmt, "M": m, "N": n - n % 4 if ws else n, "K": k, "ws": ws}
    if kind == "ffn":
        dim = 256 * rng.randint(2, 16)
        return {"kind": "ffn", "fmt": fmt, "M": rng.randint(1, 16), "dim": dim, "ffn": 256 * rng.randint(4, 44)}
    kv = rng.choice([1, 2, 4, 8])
    group = rng.choice([1, 2, 3, 4, 7, 8]) if kv <= 4 else rng.choice([1, 2, 3, 4])
    d = rng.choice([64, 64, 128])
    if kind == "prompt_attention":
        return {"kind": kind, "heads": kv * group, "kv_heads": kv, "head_dim": d, "M": _log_int(rng, 17, 2048),
                "pos": rng.choice([0, 0, _log_int(rng, 1, 2048)])}
    if kind == "token_attention":
        return {"kind": kind, "heads": kv * group, "kv_heads": kv, "head_dim": d, "T": _log_int(rng, 1, 16384)}
    prompt = kind == "prompt"
    m = _log_int(rng, 17, 2048) if prompt else rng.choice([1, rng.randint(2, 16)])
    pos = rng.choice([0, rng.randint(1, 1000)]) if prompt else rng.randint(0, 2000)
    return {"kind": kind, "layers": rng.randint(1, 4), "dim": 256 * rng.randint(2, 12), "heads": kv * group,
            "kv_heads": kv, "head_dim": d, "ffn": 256 * rng.randint(4, 32), "vocab": _log_int(rng, 4000, 64000),
            "fmt": fmt if d * kv * group % 256 == 0 else rng.choice(["q8_0", "q4_0", "q5_0", "fp16"]),
            "head": rng.choice(["q6_k", "q8_0"]), "table": "q8_0", "M": m, "pos": pos,
            "max_seq": pos + m + rng.randint(0, 512)}


# --------------------------------------------------------------------------- weights

def _gen(seed, *what):
    s = seed & 0xFFFFFFFF
    for w in what:
        s = (s * 1000003 + int(w) + 0x9E37) & 0x7FFFFFFFFFFF
    return torch.Generator(device="cuda").manual_seed(s)


def _half_bytes(x):
    return x.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _safe_inv(x):
    return torch.where(x > 0, 1.0 / torch.where(x > 0, x, torch.ones_like(x)), torch.zeros_like(x))


def _quantize(fmt, x):
    """GGUF bytes of the rows x [n, K] (float32, on the GPU), [n, row bytes]."""
    n, K = x.shape
    if fmt == "fp16":
        return x.to(torch.float16).view(torch.uint8)
    be, bb = BLOCK[fmt]
    b = x.reshape(-1, be)
    if fmt in ("q8_0", "q4_0", "q5_0"):
        top = {"q8_0": 127.0, "q4_0": 8.0, "q5_0": 16.0}[fmt]
        d = b.abs().amax(1) / top
        q = torch.round(b * _safe_inv(d)[:, None])
        if fmt == "q8_0":
            parts = [_half_bytes(d), q.clamp(-128, 127).to(torch.int8).view(torch.uint8)]
        elif fmt == "q4_0":  # element i: the low (even i) or high nibble of byte i / 2
            q = (q + 8).clamp(0, 15).to(torch.uint8)
            parts = [_half_bytes(d), q[:, 0::2] | (q[:, 1::2] << 4)]
        else:  # low nibbles of elements i and i + 16 in byte i, the fifth bits in a 32-bit mask
            q = (q + 16).clamp(0, 31).to(torch.uint8)
            bits = (q >> 4).reshape(-1, 4, 8) << torch.arange(8, device=x.device, dtype=torch.uint8)
            lo = q & 15
            parts = [_half_bytes(d), bits.sum(2, dtype=torch.uint8), lo[:, :16] | (lo[:, 16:] << 4)]
        return torch.cat(parts, 1).reshape(n, -1)
    if fmt == "q4_k":
        s = b.reshape(-1, 8, 32)
        low = s.amin(2).clamp(max=0)
        scale, off = (s.amax(2) - low) / 15, -low
        d, dmin = (scale.amax(1) / 63).to(torch.float16).float(), (off.amax(1) / 63).to(torch.float16).float()
        sc = torch.round(scale * _safe_inv(d)[:, None]).clamp(0, 63)
        mn = torch.round(off * _safe_inv(dmin)[:, None]).clamp(0, 63)
        q = torch.round((s + (dmin[:, None] * mn)[:, :, None]) * _safe_inv(d[:, None] * sc)[:, :, None])
        q = q.clamp(0, 15).to(torch.uint8).reshape(-1, 4, 2, 32)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                            (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
        qs = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)
        return torch.cat([_half_bytes(d), _half_bytes(dmin), packed, qs], 1).reshape(n, -1)
    # q6_k: 16 sub-blocks of 16 with int8 scales
    s = b.reshape(-1, 16, 16)
    top = s.abs().amax(2) / 31
    d = (top.amax(1) / 127).to(torch.float16).float()
    sc = torch.round(top * _safe_inv(d)[:, None]).clamp(0, 127)
    q = (torch.round(s * _safe_inv(d[:, None] * sc)[:, :, None]) + 32).clamp(0, 63).to(torch.uint8)
    q = q.reshape(-1, 2, 4, 32)  # half, quarter, element
    ql = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    h = q >> 4
    qh = h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _half_bytes(d)],
                     1).reshape(n, -1)


def _dequantize(fmt, w, K):
    """float64 [n, K] of the rows w [n, row bytes]."""
    n = w.shape[0]
    if fmt == "fp16":
        return w.contiguous().view(torch.float16).double()
    bb = BLOCK[fmt][1]
    b = w.reshape(-1, bb)

    def half(a):
        return b[:, a:a + 2].contiguous().view(torch.float16).double()

    if fmt == "q8_0":
        x = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q4_0":
        q = b[:, 2:]
        x = half(0) * (torch.stack([q & 15, q >> 4], 2).reshape(-1, 32).double() - 8)
    elif fmt == "q5_0":
        bits = (b[:, 2:6, None] >> torch.arange(8, device=w.device, dtype=torch.uint8)) & 1
        q = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1) | (bits.reshape(-1, 32) << 4)
        x = half(0) * (q.double() - 16)
    elif fmt == "q4_k":
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        x = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    else:
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        x = (half(208) * sc)[:, :, None] * (q.reshape(-1, 16, 16).double() - 32)
    return x.reshape(n, K)


def _weights(fmt, N, K, seed, *what):
    """Quantized N(0, 0.02) weights, [N, row bytes]."""
    g = _gen(seed, *what)
    out = torch.empty(N, K // BLOCK[fmt][0] * BLOCK[fmt][1], dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 25) // K)
    for a in range(0, N, step):
        n = min(step, N - a)
        out[a:a + n] = _quantize(fmt, torch.randn(n, K, generator=g, device="cuda") * 0.02)
    return out


def _randn(seed, what, *shape):
    return torch.randn(*shape, generator=_gen(seed, what), device="cuda")


def _times(x, fmt, w, K):
    """x [M, K] float64 times the rows of w, [M, n]."""
    step = max(1, (1 << 26) // K)
    return torch.cat([x @ _dequantize(fmt, w[a:a + step], K).t() for a in range(0, w.shape[0], step)], 1)


def _row_bytes(fmt, K):
    return K // BLOCK[fmt][0] * BLOCK[fmt][1]


# --------------------------------------------------------------------------- the decode step's parts

class _Address:
    """Device memory the decoder owns, for torch.as_tensor; the tensor's storage keeps the owner alive."""

    def __init__(self, owner, address, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 2}


def _mats(c):
    D, Q, KV, F = c["dim"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["ffn"]
    return {"q": (Q, D), "k": (KV, D), "v": (KV, D), "o": (D, Q), "gate": (F, D), "up": (F, D), "down": (D, F)}


def _layer(c, seed, i):
    mats = {n: _weights(c["fmt"], N, K, seed, 10 + i, j) for j, (n, (N, K)) in enumerate(_mats(c).items())}
    norms = [1 + 0.1 * _randn(seed, 1000 + 2 * i + j, c["dim"]) for j in range(2)]
    past = [_randn(seed, 2000 + 2 * i + j, c["pos"], c["kv_heads"] * c["head_dim"]) for j in range(2)]
    return mats, norms, past


def _ids(c, seed):
    return torch.randint(0, c["vocab"], (c["M"],), generator=_gen(seed, 3), device="cuda", dtype=torch.int32)


def _prepare_step(c, seed):
    dec = cri.Decoder(c["layers"], c["dim"], c["heads"], c["kv_heads"], c["head_dim"], c["ffn"], c["vocab"],
                      c["max_seq"], max_batch=max(16, c["M"]), rms_norm_eps=EPS, rope_theta=THETA)
    kv, rows = c["kv_heads"] * c["head_dim"], []
    for i in range(c["layers"]):
        mats, norms, past = _layer(c, seed, i)
        dec.set_layer(i, norms[0], norms[1], **{n: (c["fmt"], w) for n, w in mats.items()})
        for address, p in zip(dec.kv_cache(i), past):
            cache = torch.as_tensor(_Address(dec, address, (c["max_seq"], kv)), device="cuda")
            cache[:c["pos"]] = p
            rows.append(cache[c["pos"]:c["pos"] + c["M"]])
    dec.set_embedding(c["table"], _weights(c["table"], c["vocab"], c["dim"], seed, 4))
    dec.set_output(1 + 0.1 * _randn(seed, 5, c["dim"]), (c["head"], _weights(c["head"], c["vocab"], c["dim"], seed, 6)))
    s = {"case": c, "dec": dec, "ids": _ids(c, seed), "rows": rows}
    if c["kind"] == "prompt":
        s["logits"] = torch.empty(c["vocab"], device="cuda")
    else:
        s["logits"] = torch.empty(c["M"], c["vocab"], device="cuda")
        s["next"] = torch.empty(c["M"], dtype=torch.int32, device="cuda")
        stream = torch.cuda.Stream()
        dec.set_position(c["pos"])
        torch.cuda.synchronize()
        dec.capture(s["ids"], c["M"], s["logits"], s["next"], stream=stream)
    return s


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _silu(x):
    return x * torch.sigmoid(x)


def _rope(x, pos, heads, d):
    """Pairs (2i, 2i + 1) of each head turned by (position) * theta^(-2i / d); the angle in float32, as GGUF
    runtimes (and the reference) form it."""
    e = torch.arange(0, d, 2, device="cuda", dtype=torch.float32) / d
    freq = (1.0 / (THETA ** e.double()).float())
    at = torch.arange(pos, pos + x.shape[0], device="cuda", dtype=torch.float32)
    ang = (at[:, None] * freq[None, :]).double()[:, None, :]
    x = x.reshape(x.shape[0], heads, d // 2, 2)
    a, b = x[..., 0], x[..., 1]
    return torch.stack([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], 3).reshape(x.shape[0], -1)


def _attention(q, k, v, heads, kv_heads, d, pos):
    """q [M, heads * d] at positions pos .. over k, v [pos + M, kv_heads * d], causal, float64."""
    M, T, G = q.shape[0], k.shape[0], heads // kv_heads
    hidden = torch.arange(T, device="cuda")[None, :] > pos + torch.arange(M, device="cuda")[:, None]
    out = []
    for h in range(heads):
        g = slice(h // G * d, (h // G + 1) * d)
        s = (q[:, h * d:(h + 1) * d] @ k[:, g].t()) / math.sqrt(d)
        out.append(torch.softmax(s.masked_fill(hidden, float("-inf")), 1) @ v[:, g])
    return torch.cat(out, 1)


def _exact_step(c, seed):
    table = _weights(c["table"], c["vocab"], c["dim"], seed, 4)
    x = _dequantize(c["table"], table[_ids(c, seed).long()], c["dim"])
    f, H, KV, d, rows = c["fmt"], c["heads"], c["kv_heads"], c["head_dim"], []
    for i in range(c["layers"]):
        mats, norms, past = _layer(c, seed, i)
        n = _rms(x, norms[0])
        q, k, v = (_times(n, f, mats[m], c["dim"]) for m in "qkv")
        q, k = _rope(q, c["pos"], H, d), _rope(k, c["pos"], KV, d)
        rows += [k, v]
        ctx = _attention(q, torch.cat([past[0].double(), k]), torch.cat([past[1].double(), v]), H, KV, d, c["pos"])
        x = x + _times(ctx, f, mats["o"], H * d)
        n = _rms(x, norms[1])
        act = _silu(_times(n, f, mats["gate"], c["dim"])) * _times(n, f, mats["up"], c["dim"])
        x = x + _times(act, f, mats["down"], c["ffn"])
    if c["kind"] == "prompt":
        x = x[-1:]
    n = _rms(x, 1 + 0.1 * _randn(seed, 5, c["dim"]))
    logits = _times(n, c["head"], _weights(c["head"], c["vocab"], c["dim"], seed, 6), c["dim"])
    return (logits[0], rows) if c["kind"] == "prompt" else (logits, None, rows)


# --------------------------------------------------------------------------- prepare, run

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("step", "prompt"):
        return _prepare_step(c, seed)
    s = {"case": c}
    if kind == "matmul":
        s["A"], s["B"] = _randn(seed, 1, c["M"], c["K"]), _weights(c["fmt"], c["N"], c["K"], seed, 2)
        s["C"] = torch.empty(c["M"], c["N"], device="cuda")
        if c["ws"]:
            need = cri.matmul_workspace_bytes(c["fmt"], c["M"], c["N"], c["K"])
            s["work"] = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    elif kind == "ffn":
        D, F, M = c["dim"], c["ffn"], c["M"]
        s["hidden"], s["residual"], s["norm"] = (_randn(seed, 1, M, D), _randn(seed, 2, M, D),
                                                 1 + 0.1 * _randn(seed, 3, D))
        s["gate_up"], s["down"] = _weights(c["fmt"], 2 * F, D, seed, 4), _weights(c["fmt"], D, F, seed, 5)
        s["hidden_out"], s["out"] = torch.empty(M, D, device="cuda"), torch.empty(M, D, device="cuda")
        s["act"] = torch.empty(M, 2 * F, device="cuda")
    elif kind == "prompt_attention":
        H, KV, d, T = c["heads"], c["kv_heads"], c["head_dim"], c["pos"] + c["M"]
        s["qkv"] = _randn(seed, 1, c["M"], (H + 2 * KV) * d)
        s["k"], s["v"] = _randn(seed, 2, T, KV * d), _randn(seed, 3, T, KV * d)
        s["out"] = torch.empty(c["M"], H * d, device="cuda")
        need = cri.prefill_attention_workspace_bytes(c["M"], H, KV, d, T)
        s["work"] = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    else:
        H, KV, d, T = c["heads"], c["kv_heads"], c["head_dim"], c["T"]
        s["q"], s["k"], s["v"] = _randn(seed, 1, H * d), _randn(seed, 2, T, KV * d), _randn(seed, 3, T, KV * d)
        s["out"] = torch.empty(H * d, device="cuda")
        need = cri.decode_attention_workspace_size(H, KV, d, T)
        s["work"] = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "matmul":
        if c["ws"]:
            cri.matmul_ws(c["fmt"], s["A"], s["B"], s["C"], c["M"], c["N"], c["K"], s["work"])
        else:
            cri.matmul(c["fmt"], s["A"], s["B"], s["C"], c["M"], c["N"], c["K"])
        return s["C"]
    if kind == "ffn":
        D, F, M, act = c["dim"], c["ffn"], c["M"], s["act"]
        cri.matmul_rmsnorm(c["fmt"], s["hidden"], s["residual"], s["norm"], s["hidden_out"], s["gate_up"], act, M, 2 * F,
                           D, EPS)
        cri.matmul_swiglu(c["fmt"], act, act.data_ptr() + 4 * F, 2 * F, s["down"], s["out"], M, D, F)
        return s["out"], s["hidden_out"]
    if kind == "prompt_attention":
        H, KV, d = c["heads"], c["kv_heads"], c["head_dim"]
        cri.prefill_attention(s["qkv"], (H + 2 * KV) * d, s["k"], s["v"], s["out"], c["M"], H, KV, d, c["pos"],
                              1.0 / math.sqrt(d), s["work"])
        return s["out"]
    if kind == "token_attention":
        d = c["head_dim"]
        cri.fused_decode_attention_ws(s["q"], s["k"], s["v"], s["out"], c["heads"], c["kv_heads"], d, c["T"],
                                      1.0 / math.sqrt(d), s["work"])
        return s["out"]
    dec = s["dec"]
    dec.set_position(c["pos"])
    if kind == "prompt":
        dec.prefill(s["ids"], c["M"], s["logits"])
        return s["logits"], s["rows"]
    dec.replay()
    return s["logits"], s["next"], s["rows"]


# --------------------------------------------------------------------------- work, tolerance, exact

def work(case):
    c, kind = case, case["kind"]
    if kind == "matmul":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": N * _row_bytes(c["fmt"], K) + 4 * M * (K + N), "flops": 2 * M * N * K}
    if kind == "ffn":
        D, F, M = c["dim"], c["ffn"], c["M"]
        return {"bytes": 2 * F * _row_bytes(c["fmt"], D) + D * _row_bytes(c["fmt"], F) + 4 * (4 * M * D + D),
                "flops": 6 * M * D * F}
    H, KV, d = c["heads"], c["kv_heads"], c["head_dim"]
    if kind == "token_attention":
        return {"bytes": 4 * (2 * H * d + 2 * c["T"] * KV * d), "flops": 4 * H * d * c["T"]}
    M, pos = c["M"], c["pos"]
    seen = M * pos + M * (M + 1) // 2  # (row, position) pairs
    if kind == "prompt_attention":
        return {"bytes": 4 * (2 * M * H * d + 2 * (pos + M) * KV * d), "flops": 4 * H * d * seen}
    params = sum(N * K for N, K in _mats(c).values())
    layer = sum(N * _row_bytes(c["fmt"], K) for N, K in _mats(c).values()) + 8 * c["dim"] + 8 * (pos + 2 * M) * KV * d
    rows = 1 if kind == "prompt" else M
    return {"bytes": c["layers"] * layer + c["vocab"] * _row_bytes(c["head"], c["dim"]) + 4 * rows * c["vocab"]
            + M * _row_bytes(c["table"], c["dim"]),
            "flops": c["layers"] * (2 * M * params + 4 * H * d * seen) + 2 * rows * c["vocab"] * c["dim"]}


def tolerance(case):
    """About four times the distance from float64 that these paths show."""
    c, kind = case, case["kind"]
    if kind == "matmul" and c["M"] > 16:
        return {"rel": 2e-3}  # fp16 operands, fp32 sums: 2.9e-4 (one rounding of a weight) to 5.2e-4 (q4_k)
    if kind == "prompt":
        return {"rel": 4e-3 + 1e-3 * c["layers"]}  # those products compounded: 4.6e-3 after 16 layers
    if kind == "step":
        return {"rel": 1.2e-5, "differ": 0.0}  # fp32 throughout: 3.1e-6 after 16 layers
    return {"rel": 4e-6}  # one or two fp32 products, or an fp32 softmax between two


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("step", "prompt"):
        return _exact_step(c, seed)
    if kind == "matmul":
        return _times(_randn(seed, 1, c["M"], c["K"]).double(), c["fmt"], _weights(c["fmt"], c["N"], c["K"], seed, 2),
                      c["K"])
    if kind == "ffn":
        D, F, M = c["dim"], c["ffn"], c["M"]
        h = _randn(seed, 1, M, D) + _randn(seed, 2, M, D)  # the residual stream is float32
        gu = _times(_rms(h.double(), 1 + 0.1 * _randn(seed, 3, D)), c["fmt"],
                    _weights(c["fmt"], 2 * F, D, seed, 4), D)
        return _times(_silu(gu[:, :F]) * gu[:, F:], c["fmt"], _weights(c["fmt"], D, F, seed, 5), F), h.double()
    H, KV, d = c["heads"], c["kv_heads"], c["head_dim"]
    if kind == "token_attention":
        q, k, v = _randn(seed, 1, 1, H * d), _randn(seed, 2, c["T"], KV * d), _randn(seed, 3, c["T"], KV * d)
        return _attention(q.double(), k.double(), v.double(), H, KV, d, c["T"] - 1)[0]
    T = c["pos"] + c["M"]
    q = _randn(seed, 1, c["M"], (H + 2 * KV) * d)[:, :H * d]
    return _attention(q.double(), _randn(seed, 2, T, KV * d).double(), _randn(seed, 3, T, KV * d).double(), H, KV, d,
                      c["pos"])
