"""The work whose speed this repository is measured by, case by case.

Every case is one call (or one chain of calls) through the public entry points,
at the sizes of the repository's own configurations: the linears, the delta-net,
the attention of an ~8B hybrid (d_model 4096, 32 q / 8 kv heads of 128, 32
delta-net heads of 128 x 128, SwiGLU 12288), and a whole generation request on
a model of that width. A case's numbers do not depend on the GPU; prepare()
makes its inputs from the seed alone.
"""
import functools
import math
from dataclasses import replace

import numpy as np
import torch

import hero_amd
from hero_amd._lib import AttnDecodeArgs, AttnPagedArgs, GdnDecodeArgs, check, lib

Q4_K, Q5_K, Q6_K = 12, 13, 14  # ggml types
BLOCK_BYTES = {Q4_K: 144, Q5_K: 176, Q6_K: 210}  # per 256 weights
CONV_W = 4
EPS = 1e-6
ROPE_BASE = 1e6


def listed():
    return [
        # A Q8_0 projection of one decoded token (4096-row out-projection): the smallest call, latency and launches count.
        {"name": "decode_linear_q8", "kind": "linear_q8", "m": 1, "n": 4096, "k": 4096},
        # The same kind of product for sixteen sequences decoded together (a projection to the FFN width).
        {"name": "batch_linear_q8", "kind": "linear_q8", "m": 16, "n": 12288, "k": 4096},
        # A prompt's rows through a Q8_0 FFN projection; a prompt is rarely a whole number of tiles.
        {"name": "prefill_linear_q8", "kind": "linear_q8", "m": 1000, "n": 12288, "k": 4096},
        # One decoded token through a Q4_K projection of a Q4_K_M checkpoint (FFN gate or up).
        {"name": "decode_linear_q4k", "kind": "linear_kq", "type": Q4_K, "m": 1, "n": 12288, "k": 4096},
        # A prompt through the checkpoint's Q4_K projections (ssm_out, gate, up).
        {"name": "prefill_linear_q4k", "kind": "linear_kq", "type": Q4_K, "m": 509, "n": 4096, "k": 4096},
        # A prompt through its Q5_K projections (attn_qkv, attn_output), which take fp32 activations.
        {"name": "prefill_linear_q5k", "kind": "linear_kq", "type": Q5_K, "m": 256, "n": 4096, "k": 4096},
        # A prompt through its Q6_K down projection.
        {"name": "prefill_linear_q6k", "kind": "linear_kq", "type": Q6_K, "m": 512, "n": 4096, "k": 12288},
        # The delta-net layer body of one decode step of sixteen sequences.
        {"name": "gdn_decode_b16", "kind": "gdn_decode", "b": 16, "hk": 32, "hv": 32},
        # The delta-net layer body over one prefill chunk, token-serial (the exact form).
        {"name": "gdn_prefill_1024", "kind": "gdn_prefill", "t": 1024, "hk": 32, "hv": 32, "chunked": False},
        # One decoded token's attention over a long context, fp32 cache (the reference's precision).
        {"name": "attn_decode_8k", "kind": "attn_decode", "b": 1, "ctx": 8192, "window": 0, "cache": "fp32", "dh": 128},
        # A prefill chunk's attention in the middle of a prompt: 1024 rows after 1024 cached ones.
        {"name": "attn_prefill_1024", "kind": "attn_prefill", "t": 1024, "past": 1024, "window": 0, "dh": 128},
        # A whole request on a four-layer model of the 8B width: prompt in, greedy tokens and logits out.
        {"name": "generate", "kind": "generate", "prompt": 300, "steps": 16, "mix": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: rows from one token to a prefill chunk, the
    row lengths and heights of the configurations and ragged ones, contexts from
    a short chat to 32k, every cache type and window."""
    kind = rng.choice(["linear_q8", "linear_q8", "linear_kq", "linear_kq", "linear_kq", "gdn_decode", "gdn_prefill", "attn_decode", "attn_decode",
                       "attn_prefill", "generate"])
    if kind == "linear_q8":
        k = rng.choice([1024, 2560, 2816, 4096, 4096, 8192, 12288])
        n = rng.choice([4096, 10240, 12288, 16448, _log(rng, 1000, 16000)])
        return {"kind": kind, "m": min(_log(rng, 1, 1024), (1000 * 12288 * 4096) // (n * k)), "n": n, "k": k}
    if kind == "linear_kq":
        t = rng.choice([Q4_K, Q5_K, Q6_K])
        k = rng.choice([1024, 2816, 4096, 4096, 8192, 12288])
        n = rng.choice([4096, 8192, 12288, _log(rng, 1000, 12000)])
        most = (256 * 4096 * 4096 if t == Q5_K else 512 * 4096 * 12288) // (n * k)
        return {"kind": kind, "type": t, "m": max(1, min(_log(rng, 1, 700), most)), "n": n, "k": k}
    hk, hv = rng.choice([(32, 32), (16, 16), (16, 32), (8, 8)])
    if kind == "gdn_decode":
        return {"kind": kind, "b": rng.randint(1, 16), "hk": hk, "hv": hv}
    if kind == "gdn_prefill":
        return {"kind": kind, "t": _log(rng, 16, 1024), "hk": hk, "hv": hv, "chunked": rng.random() < 0.3}
    if kind == "attn_decode":
        cache, b = rng.choice(["fp32", "fp16", "q8"]), rng.choice([1, 1, 2, rng.randint(3, 16)])
        dh = rng.choice([128, 128, 256]) if cache != "q8" else 128
        return {"kind": kind, "b": b, "ctx": _log(rng, 100, min(32768, 65536 // b)), "window": rng.choice([0, 0, 1024]), "cache": cache, "dh": dh}
    if kind == "attn_prefill":
        return {"kind": kind, "t": _log(rng, 16, 1024), "past": rng.choice([0, rng.randint(1, 1024)]), "window": rng.choice([0, 0, 512]),
                "dh": rng.choice([128, 128, 256])}
    return {"kind": kind, "prompt": _log(rng, 8, 300), "steps": rng.randint(1, 16), "mix": rng.choice([0, 1])}


# ---- shared pieces ---------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (seed + 1))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device="cuda")


def _p(t):
    return t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _act_parts(act, m, k):
    """A quantized activation buffer as its int8 values and its fp32 scales."""
    return act[: m * k].view(torch.int8).view(m, k), act[m * k: m * k + m * (k // 32) * 4].view(torch.float32).view(m, k // 32)


def _quant_q8_0(x):
    """The activation quantizer in its own (fp32) steps: int values and fp16-rounded scales (ties away from zero), both as float64."""
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1) / torch.full((), 127.0, device=x.device)  # a tensor: division by a number multiplies by its reciprocal
    inv = torch.where(d > 0, torch.ones_like(d) / d, torch.zeros_like(d))
    v = (b * inv[..., None]).double()
    d16 = ((d.view(torch.int32) + 0x1000) & -0x2000).view(torch.float32)
    return torch.sign(v) * torch.floor(v.abs() + 0.5), d16.double()


# ---- Q8_0 linear: activation quantizer + matvec / matmul --------------------------------------------
def _q8_weight(g, n, k):
    """N(0, 0.02) weights as Q8_0: int8 [n, k/32, 32] and fp16 scales [n, k/32]."""
    w = _randn(g, n, k // 32, 32) * 0.02
    d = (w.abs().amax(-1) / 127.0).half()
    return torch.clamp(torch.round(w / d.float()[..., None]), -127, 127).to(torch.int8), d


def _q8_blocks(q, d):
    return torch.cat([d.view(torch.uint8).view(*d.shape, 2), q.view(torch.uint8)], dim=-1).contiguous()


def _prepare_linear_q8(c, g):
    m, n, k = c["m"], c["n"], c["k"]
    blocks = _q8_blocks(*_q8_weight(g, n, k))
    packed = _bytes(lib.hero_q8_0_packed_bytes(n, k))
    check(lib.hero_q8_0_pack(_p(blocks), _p(packed), n, k, 0, n, _stream()))
    torch.cuda.synchronize()
    return {"w": packed, "x": _randn(g, m, k), "act": _bytes(lib.hero_q8_0_act_bytes(m, k)), "y": torch.empty(m, n, device="cuda")}


def _run_linear_q8(s, c):
    m, n, k, st = c["m"], c["n"], c["k"], _stream()
    check(lib.hero_q8_0_quantize(_p(s["x"]), _p(s["act"]), m, k, st))
    if m == 1:
        check(lib.hero_q8_0_gemv(_p(s["w"]), _p(s["act"]), _p(s["y"]), None, n, k, st))
    else:
        check(lib.hero_q8_0_gemm(_p(s["w"]), _p(s["act"]), _p(s["y"]), None, m, n, k, st))
    return s["y"]


def _exact_linear_q8(c, g):
    q, d = _q8_weight(g, c["n"], c["k"])
    x = _randn(g, c["m"], c["k"])
    w = (q.double() * d.double()[..., None]).view(c["n"], c["k"])
    xq, xd = _quant_q8_0(x)
    return (xq * xd[..., None]).view(c["m"], c["k"]) @ w.T


# ---- K-quant linear: Q4_K / Q6_K on Q8_K activations, Q5_K on fp32 -----------------------------------
def _kq_blocks(g, t, n, k):
    """Random GGUF super-blocks with scales of a trained checkpoint's size; the mins centre the weights."""
    nb = n * (k // 256)
    w = torch.randint(0, 256, (nb, BLOCK_BYTES[t]), dtype=torch.uint8, device="cuda", generator=g)
    d = torch.rand(nb, device="cuda", generator=g) * 1e-4 + 5e-5
    half = lambda v: v.half().view(torch.uint8).view(nb, 2)  # noqa: E731
    if t == Q6_K:
        w[:, 208:210] = half(d)
    else:
        w[:, 0:2] = half(d)
        w[:, 2:4] = half(d * (7.5 if t == Q4_K else 15.5))
    return w


def _kq_dequant(w, t, n, k):
    """The GGUF blocks as float64 weights [n, k]."""
    f16 = lambda lo: w[:, lo:lo + 2].contiguous().view(torch.float16).double()  # noqa: E731  [nb, 1]
    if t == Q6_K:
        ql, qh, sc = w[:, :128].view(-1, 2, 2, 32), w[:, 128:192].view(-1, 2, 32), w[:, 192:208].contiguous().view(torch.int8).double()
        parts = []
        for h in range(2):  # halves of 128; sub-blocks of 32 in order
            for j in range(4):
                lo = (ql[:, h, j % 2] >> (4 * (j // 2))) & 15
                parts.append((lo | (((qh[:, h] >> (2 * j)) & 3) << 4)).double() - 32)
        q = torch.stack(parts, 1).view(-1, 16, 16)
        return (q * sc[..., None] * f16(208)[..., None]).view(n, k)
    s = w[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = w[:, -128:].view(-1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
    if t == Q5_K:
        bit = torch.arange(8, device=w.device, dtype=torch.uint8).view(1, 8, 1)
        q = q | (((w[:, 16:48].view(-1, 1, 32) >> bit) & 1) << 4)
    return (f16(0)[..., None] * sc[..., None] * q.double() - f16(2)[..., None] * mn[..., None]).view(n, k)


def _prepare_linear_kq(c, g):
    t, m, n, k = c["type"], c["m"], c["n"], c["k"]
    blocks = _kq_blocks(g, t, n, k)
    packed = _bytes(lib.hero_kquant_packed_bytes(t, n, k))
    check(lib.hero_kquant_pack(t, _p(blocks), _p(packed), n, k, _stream()))
    torch.cuda.synchronize()
    act = _bytes(lib.hero_q8_K_act_bytes(m, k)) if t != Q5_K else None
    return {"w": packed, "x": _randn(g, m, k), "act": act, "y": torch.empty(m, n, device="cuda")}


def _run_linear_kq(s, c):
    t, m, n, k, st = c["type"], c["m"], c["n"], c["k"], _stream()
    if t == Q5_K:
        check(lib.hero_q5_K_gemm(_p(s["w"]), _p(s["x"]), _p(s["y"]), m, n, k, st))
    else:
        check(lib.hero_q8_K_quantize(_p(s["x"]), _p(s["act"]), m, k, st))
        check(lib.hero_kquant_gemm(t, _p(s["w"]), _p(s["act"]), _p(s["y"]), m, n, k, st))
    return s["y"]


def _exact_linear_kq(c, g):
    t, m, n, k = c["type"], c["m"], c["n"], c["k"]
    w = _kq_dequant(_kq_blocks(g, t, n, k), t, n, k)
    x = _randn(g, m, k)
    if t == Q5_K:
        return x.double() @ w.T
    b = x.view(m, -1, 256)  # Q8_K: -127 / (the element of largest magnitude), round to nearest even
    top = torch.gather(b, 2, b.abs().argmax(-1, keepdim=True))
    inv = torch.full_like(top, -127.0) / top
    q = torch.clamp(torch.round(b * inv), max=127).double()
    return (q * (torch.ones_like(inv) / inv).double()).view(m, k) @ w.T


# ---- gated delta-net layer body ----------------------------------------------------------------------
def _gdn_inputs(c, g):
    hk, hv, rows = c["hk"], c["hv"], c.get("b") or c["t"]
    seqs = c.get("b", 1)
    cc = 2 * hk * 128 + hv * 128
    stride = cc + hv * 128 + 2 * hv  # [qkv | z | beta | alpha]
    first = torch.randint(8, 2000, (seqs,), device="cuda", generator=g, dtype=torch.int32)
    return {
        "proj": _randn(g, rows, stride), "taps": _randn(g, cc, CONV_W) * 0.5, "hist": _randn(g, seqs, CONV_W, cc),
        "state": _randn(g, seqs, hv, 128, 128) * 0.05, "dt": _randn(g, hv) * 0.5,
        "decay": -torch.exp(torch.rand(hv, device="cuda", generator=g) * 3 - 2), "gamma": 1 + 0.1 * _randn(g, 128),
        "pos": first if "b" in c else first + torch.arange(rows, device="cuda", dtype=torch.int32),
    }


def _prepare_gdn(c, g):
    s = _gdn_inputs(c, g)
    hk, hv, rows = c["hk"], c["hv"], s["proj"].shape[0]
    cc, stride = s["taps"].shape[0], s["proj"].shape[1]
    s["act"], s["out"] = _bytes(lib.hero_q8_0_act_bytes(rows, hv * 128)), torch.empty(rows, hv * 128, device="cuda")
    s["args"] = GdnDecodeArgs(_p(s["proj"]), stride, cc, cc + hv * 128, cc + hv * 128 + hv, _p(s["taps"]), _p(s["hist"]), _p(s["state"]), _p(s["dt"]),
                              _p(s["decay"]), _p(s["gamma"]), EPS, _p(s["pos"]), _p(s["act"]), _p(s["out"]), rows, hk, hv, 128, 128, CONV_W)
    if "t" in c:
        s["work_bytes"] = lib.hero_gdn_prefill_work_bytes(rows, hk, hv)
        s["work"] = _bytes(s["work_bytes"])
    return s


def _run_gdn(s, c):
    if "t" in c:
        f = lib.hero_gdn_prefill_chunked if c["chunked"] else lib.hero_gdn_prefill
        check(f(s["args"], _p(s["work"]), s["work_bytes"], _stream()))
    else:
        check(lib.hero_gdn_decode(s["args"], _stream()))
    return [s["out"], *_act_parts(s["act"], *s["out"].shape), s["state"], s["hist"]]


def _exact_gdn(c, g):
    s = {k: v if k == "pos" else v.double() for k, v in _gdn_inputs(c, g).items()}
    hk, hv = c["hk"], c["hv"]
    kw, cc = hk * 128, s["taps"].shape[0]
    rows, state, hist, outs = s["proj"].shape[0], s["state"], s["hist"], []
    silu = lambda v: v * torch.sigmoid(v)  # noqa: E731
    norm = lambda v: v / torch.clamp(torch.sqrt((v * v).sum(-1, keepdim=True)), min=1e-6)  # noqa: E731
    seq = torch.arange(hist.shape[0], device="cuda")  # value head h reads key head h % hk
    for i in range(rows if "t" in c else 1):
        p = s["proj"][i:i + 1] if "t" in c else s["proj"]
        pos = s["pos"][i:i + 1].long() if "t" in c else s["pos"].long()
        u = s["taps"][:, CONV_W - 1] * p[:, :cc]
        for j in range(CONV_W - 1):
            u = u + s["taps"][:, j] * hist[seq, (pos - (CONV_W - 1) + j) % CONV_W]
        hist[seq, pos % CONV_W] = p[:, :cc]
        u = silu(u)
        q = norm(u[:, :kw].view(-1, hk, 128)) / math.sqrt(128.0)
        k = norm(u[:, kw:2 * kw].view(-1, hk, 128))
        q, k = (v.repeat(1, hv // hk, 1) for v in (q, k))
        v = u[:, 2 * kw:].view(-1, hv, 128)
        beta = torch.sigmoid(p[:, cc + hv * 128:cc + hv * 128 + hv])
        gate = torch.exp(s["decay"] * torch.nn.functional.softplus(p[:, cc + hv * 128 + hv:] + s["dt"]))
        state *= gate[..., None, None]
        delta = (v - (state * k[..., None]).sum(-2)) * beta[..., None]
        state += k[..., None] * delta[..., None, :]
        o = (state * q[..., None]).sum(-2)
        o = s["gamma"] * o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS)
        outs.append(o.reshape(-1, hv * 128) * silu(p[:, cc:cc + hv * 128]))
    return [torch.cat(outs), None, None, state, hist]


# ---- gated GQA attention -----------------------------------------------------------------------------
HQ, HKV = 32, 8


@functools.lru_cache(maxsize=4)
def _rope(dh, positions):
    """cos / sin [positions][dh/2][2] of the first quarter of the planes, as a loader lays them out once"""
    inv = np.zeros(dh // 2, np.float32)
    inv[: dh // 8] = (ROPE_BASE ** (-2.0 * np.arange(dh // 8) / dh)).astype(np.float32)
    angle = (np.arange(positions, dtype=np.float32)[:, None] * inv).astype(np.float32)
    return torch.from_numpy(np.stack([np.cos(angle), np.sin(angle)], -1)).cuda()


def _attn_shape(c):
    b, ctx = (c["b"], c["ctx"]) if "b" in c else (1, c["past"] + c["t"])
    rows = c.get("t") or b
    return b, rows, ctx, -(-ctx // 64) * 64, c["dh"], c.get("cache", "fp32")


def _attn_inputs(c, g):
    b, rows, ctx, span, dh, cache = _attn_shape(c)
    kw = HKV * dh
    s = {"proj": _randn(g, rows, 2 * HQ * dh + 2 * kw), "gq": 1 + 0.1 * _randn(g, dh), "gk": 1 + 0.1 * _randn(g, dh)}
    if "t" in c:
        s["pos"] = c["past"] + torch.arange(rows, device="cuda", dtype=torch.int32)
    else:  # sequences of a batch differ a little in length
        s["pos"] = ctx - 1 - torch.randint(0, max(1, ctx // 8), (b,), device="cuda", generator=g, dtype=torch.int32)
        s["pos"][0] = ctx - 1
    if cache == "fp32":
        s["k"], s["v"] = _randn(g, b, HKV, dh, span), _randn(g, b, span, kw)
    else:
        kv = _randn(g, b * span // 64, 2, HKV, 64, dh)
        if cache == "fp16":
            s["pages"] = kv.half()
        else:
            q, d = _quant_q8_0(kv)
            n = q.shape[0]
            s["pages"] = torch.cat([q.to(torch.int8).view(n, -1).view(torch.uint8), d.half().view(n, -1).view(torch.uint8)], 1).contiguous()
    return s


def _prepare_attn(c, g):
    b, rows, ctx, span, dh, cache = _attn_shape(c)
    s = _attn_inputs(c, g)
    qw, kw = HQ * dh, HKV * dh
    s["rope"] = _rope(dh, 32768)
    s["qrot"], s["out"] = torch.empty(rows * qw, device="cuda"), torch.empty(rows, qw, device="cuda")
    s["act"] = _bytes(lib.hero_q8_0_act_bytes(rows, qw))
    fp32 = cache == "fp32"
    s["scores"] = torch.empty(rows * HQ * span, device="cuda") if fp32 else None
    a = AttnDecodeArgs(_p(s["proj"]), 2 * qw + 2 * kw, 2 * qw, 2 * qw + kw, _p(s["gq"]), _p(s["gk"]), EPS, _p(s["rope"]), _p(s["k"]) if fp32 else None,
                       _p(s["v"]) if fp32 else None, span if fp32 else 0, _p(s["pos"]), _p(s["scores"]) if fp32 else None, _p(s["qrot"]),
                       1.0 / math.sqrt(dh), c["window"], _p(s["act"]), _p(s["out"]), rows, HQ, HKV, dh)
    if not fp32:
        wb = lib.hero_attn_paged_work_bytes(span, c["window"], b, HQ, HKV, dh)
        s["work"], s["table"] = _bytes(wb), torch.randperm(b * span // 64, device="cuda", generator=g).to(torch.int32)
        a = AttnPagedArgs(a, _p(s["pages"]), _p(s["table"]), 64, span // 64, _p(s["work"]), wb, 1 if cache == "q8" else 0)
    s["args"] = a
    return s


def _run_attn(s, c):
    if "t" in c:
        check(lib.hero_attn_prefill(s["args"], _stream()))
    elif c["cache"] == "fp32":
        check(lib.hero_attn_decode(s["args"], _stream()))
    else:
        check(lib.hero_attn_decode_paged(s["args"], _stream()))
    out = [s["out"], *_act_parts(s["act"], *s["out"].shape)]
    return out + ([s["k"], s["v"]] if "k" in s else [s["pages"]])


def _exact_attn(c, g):
    b, rows, ctx, span, dh, cache = _attn_shape(c)
    s = _attn_inputs(c, g)
    qw, kw = HQ * dh, HKV * dh
    pos, rope, p = s["pos"].long(), _rope(dh, 32768).double(), s["proj"].double()

    def heads(x, gamma):  # RMSNorm and RoPE on the planes (i, i + dh/2)
        x = gamma.double() * x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
        cs, lo, hi = rope[pos][:, None], x[..., : dh // 2], x[..., dh // 2:]
        return torch.cat([lo * cs[..., 0] - hi * cs[..., 1], hi * cs[..., 0] + lo * cs[..., 1]], -1)

    qg = p[:, : 2 * qw].view(rows, HQ, 2, dh)
    q, gate = heads(qg[:, :, 0], s["gq"]), torch.sigmoid(qg[:, :, 1])
    k, v = heads(p[:, 2 * qw:2 * qw + kw].view(rows, HKV, dh), s["gk"]), p[:, 2 * qw + kw:].view(rows, HKV, dh)
    if cache == "fp32":
        keys, vals = s["k"].double().permute(0, 3, 1, 2).contiguous(), s["v"].double().view(b, span, HKV, dh)
    else:
        table = torch.randperm(b * span // 64, device="cuda", generator=g)
        if cache == "fp16":
            pages = s["pages"].double()
            k, v = k.half().double(), v.half().double()
        else:
            nq = 2 * HKV * 64 * dh
            pages = s["pages"][:, :nq].contiguous().view(torch.int8).double().view(-1, 2, HKV, 64, dh // 32, 32)
            pages = (pages * s["pages"][:, nq:].contiguous().view(torch.float16).double().view(-1, 2, HKV, 64, dh // 32, 1)).view(-1, 2, HKV, 64, dh)
            k, v = ((lambda qd: (qd[0] * qd[1][..., None]).view(rows, HKV, dh))(_quant_q8_0(x)) for x in (k, v))
        keys, vals = (pages[table][:, i].permute(0, 2, 1, 3).reshape(b, span, HKV, dh) for i in (0, 1))
    seq = torch.zeros(rows, dtype=torch.long, device="cuda") if "t" in c else torch.arange(b, device="cuda")
    keys[seq, pos], vals[seq, pos] = k, v
    outs, grp = [], HQ // HKV
    for r in range(rows):
        end, first = int(pos[r]) + 1, max(0, int(pos[r]) + 1 - c["window"]) if c["window"] else 0
        kr, vr = keys[seq[r], first:end].transpose(0, 1), vals[seq[r], first:end].transpose(0, 1)  # [HKV, keys, dh]
        w = torch.softmax((kr[:, None] * q[r].view(HKV, grp, 1, dh)).sum(-1) / math.sqrt(dh), -1) if end - first < 256 else \
            torch.softmax(torch.stack([q[r].view(HKV, grp, dh)[i] @ kr[i].T for i in range(HKV)]) / math.sqrt(dh), -1)
        outs.append(torch.stack([w[i] @ vr[i] for i in range(HKV)]).view(HQ, dh) * gate[r])
    out = [torch.stack(outs).view(rows, qw), None, None]
    if cache == "fp32":
        return out + [keys.permute(0, 2, 3, 1).contiguous(), vals.reshape(b, span, kw)]
    return out + [None]  # pages: stored 16- or 8-bit values, not computed numbers


# ---- a whole request ---------------------------------------------------------------------------------
GEN_SHAPE = replace(hero_amd.HYBRID_8B_CONFIG, layers=4, vocab=32000)  # three delta-net layers, one attention layer


@functools.lru_cache(maxsize=2)
def _checkpoint(mix):
    return hero_amd.synthetic_gguf_image(GEN_SHAPE, seed=20260101, ctx=4096, weight_mix=mix)


@functools.lru_cache(maxsize=2)
def _model(mix):
    """A server loads its checkpoint once; requests differ in their prompts and keep their own state."""
    return hero_amd.Qwen35Model.open_image(_checkpoint(mix))


def _prepare_generate(c, g):
    model = _model(c["mix"])
    ids = torch.randint(0, GEN_SHAPE.vocab, (c["prompt"],), device="cuda", generator=g).cpu().numpy().astype(np.int32)
    return {"model": model, "state": model.new_state(512), "ids": ids}


def _run_generate(s, c):
    s["state"].reset()
    logits = s["model"].forward(s["state"], ids=s["ids"])
    ids, last = s["model"].decode_greedy(s["state"], logits.argmax(), c["steps"], want_logits=True)
    return {"prefill": logits.values, "last": last.values, "ids": ids}


# ---- the interface -----------------------------------------------------------------------------------
PREPARE = {"linear_q8": _prepare_linear_q8, "linear_kq": _prepare_linear_kq, "gdn_decode": _prepare_gdn, "gdn_prefill": _prepare_gdn,
           "attn_decode": _prepare_attn, "attn_prefill": _prepare_attn, "generate": _prepare_generate}
RUN = {"linear_q8": _run_linear_q8, "linear_kq": _run_linear_kq, "gdn_decode": _run_gdn, "gdn_prefill": _run_gdn, "attn_decode": _run_attn,
       "attn_prefill": _run_attn, "generate": _run_generate}
EXACT = {"linear_q8": _exact_linear_q8, "linear_kq": _exact_linear_kq, "gdn_decode": _exact_gdn, "gdn_prefill": _exact_gdn, "attn_decode": _exact_attn,
         "attn_prefill": _exact_attn}


def prepare(case, seed):
    s = PREPARE[case["kind"]](case, _gen(seed))
    s["case"] = case
    return s


def run(state):
    return RUN[state["case"]["kind"]](state, state["case"])


def exact(case, seed):
    f = EXACT.get(case["kind"])
    return f(case, _gen(seed)) if f else None  # a quantized model has no 64-bit counterpart: each layer rounds its activations to 8 bits


def work(case):
    c, kind = case, case["kind"]
    if kind in ("linear_q8", "linear_kq"):
        m, n, k = c["m"], c["n"], c["k"]
        w = n * k * 34 // 32 if kind == "linear_q8" else n * (k // 256) * BLOCK_BYTES[c["type"]]
        return {"bytes": w + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind in ("gdn_decode", "gdn_prefill"):
        hk, hv, rows, seqs = c["hk"], c["hv"], c.get("b") or c["t"], c.get("b", 1)
        cc = 2 * hk * 128 + hv * 128
        row = 4 * (cc + 2 * hv * 128 + 2 * hv) + hv * 128 * 9 // 8
        return {"bytes": rows * row + 8 * seqs * (hv * 128 * 128 + CONV_W * cc) + 4 * cc * CONV_W, "flops": 7 * rows * hv * 128 * 128}
    if kind in ("attn_decode", "attn_prefill"):
        b, rows, ctx, span, dh, cache = _attn_shape(c)
        per = {"fp32": 4.0, "fp16": 2.0, "q8": 34 / 32}[cache]
        see = [min(p + 1, c["window"] or p + 1) for p in (range(c["past"], ctx) if "t" in c else [ctx - 1] * b)]
        keys = min(ctx, c["window"] + rows) if "t" in c and c["window"] else ctx if "t" in c else sum(see)
        row = 4 * (3 * HQ * dh + 2 * HKV * dh) + HQ * dh * 9 // 8
        return {"bytes": int(2 * keys * HKV * dh * per) + rows * row, "flops": 4 * sum(see) * HQ * dh}
    s = GEN_SHAPE
    weights = sum([3 * (16448 * 4096 + 4096 * 4096), 10240 * 4096 + 4096 * 4096, s.layers * 3 * s.ffn * s.d_model])
    head = s.vocab * s.d_model
    rows = c["prompt"] + c["steps"]
    per = 34 / 32 if c["mix"] == 0 else 0.7  # bytes per weight: Q8_0, or the tensor types of a Q4_K_M checkpoint
    return {"bytes": int((1 + c["steps"]) * per * (weights + head)), "flops": 2 * (weights * rows + head * (1 + c["steps"]))}


def tolerance(case):
    return TOLERANCE[case["kind"] if not case.get("chunked") else "gdn_chunked"]


# Four times what the fp32 sums were measured to be off their 64-bit values over the ranges of draw(); a rounding of an
# 8-bit output at its tie may fall either way. In a whole model such a tie moves a value by 1/127 of its block's largest.
TOLERANCE = {
    "linear_q8": {"rel": 1.5e-6, "max": 1.2e-5},
    "linear_kq": {"rel": 1.5e-6, "max": 1e-5},
    "gdn_decode": {"rel": 1e-6, "max": 4e-5, "differ": 1e-3},
    "gdn_prefill": {"rel": 1e-6, "max": 5e-5, "differ": 1e-3},
    "gdn_chunked": {"rel": 2.5e-6, "max": 2e-4, "differ": 2e-3},
    "attn_decode": {"rel": 2e-5, "max": 1e-4, "differ": 1e-3},
    "attn_prefill": {"rel": 4e-6, "max": 4e-5, "differ": 1e-3},
    "generate": {"rel": 0.02, "max": 0.2, "differ": 0.01},
}
