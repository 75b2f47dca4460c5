"""The work that a program with a compressed KV cache has this codec do, as cases with a size each.

A serving step compresses the new token's keys and values of every layer, a prompt's prefill compresses whole
layers, a model that attends with its own kernels decodes caches back, and one that does not attends over the
codes as they are. Every case goes through the operators of ``pitch_amd.PITCH`` (or the batch tables a program
keeps beside it) on buffers that the program owns.

Kinds of case and what their fields mean:

* append: one token's vectors of every layer into per-vector caches, one batched call (layers, heads, at = tokens
  that the caches hold already);
* append_keys: one token into every head's per-channel cache, whose last group is re-encoded (tokens = the cache's
  length after the append);
* encode: one layer's (or cache's) vectors, ``count`` of them;
* encode_keys: one layer's keys per channel, head by head when a head's tokens are no whole number of groups;
* decode: ``layers`` caches of ``count`` vectors each, batched when there are several;
* decode_keys: one layer's per-channel keys;
* attend: one query token over one layer's caches, with keys per vector, per vector with the projection's bias
  removed ("bias"), or per channel ("channel").

Sizes are those of the workloads in ``pitch_amd/workloads.py`` and ``bench.py`` (GPT-2-small: 12 heads of 64;
Qwen2.5-1.5B: 2 KV heads of 128 under 12 query heads, 28 layers; Llama-3-8B: 8 KV heads of 128 under 32 query
heads, 32 layers), with prompts and caches of ordinary and ragged lengths.
"""
from __future__ import annotations

import json
import math
from pathlib import Path

import torch

import pitch_amd as P
from pitch_amd import workloads as W

SEED = 0x50495443
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
LAYER_VECTORS = 1 << 20    # most vectors of a drawn encode or decode: 8 heads x 131072 tokens


def listed() -> list[dict]:
    return [
        # a decode step's new value vectors of all 32 layers of Llama-3-8B, a bfloat16 model
        dict(name="append_values_bf16", kind="append", method="turboQuant", layers=32, heads=8, at=1000, dim=128,
             bits=4, dtype="bfloat16"),
        # the same step's new keys of one layer, per channel: eight heads' growing groups
        dict(name="append_keys_kivi_bf16", kind="append_keys", heads=8, tokens=1000, dim=128, bits=4, group=64,
             dtype="bfloat16"),
        # prefill of an 8191-token prompt: one layer's values, bfloat16
        dict(name="prefill_values_bf16", kind="encode", method="turboQuant", count=8 * 8191, heads=8, dim=128, bits=4,
             dtype="bfloat16"),
        # a whole GPT-2 layer's values at 32768 tokens, float32, three bits
        dict(name="prefill_values_f32", kind="encode", method="turboQuant", count=12 * 32768, heads=12, dim=64,
             bits=3, dtype="float32"),
        # PolarQuant of a Qwen2.5-1.5B layer's values at 50001 tokens, float16
        dict(name="prefill_polar_f16", kind="encode", method="polarQuant", count=2 * 50001, heads=2, dim=128, bits=4,
             dtype="float16"),
        # prefill of 32768 tokens: one Llama-3-8B layer's keys per channel, bfloat16
        dict(name="prefill_keys_kivi_bf16", kind="encode_keys", heads=8, tokens=32768, dim=128, bits=4, group=64,
             dtype="bfloat16"),
        # the value caches of four Llama-3-8B layers at 131072 tokens decoded in one call, float32, three bits
        dict(name="decode_cache_f32", kind="decode", method="turboQuant", layers=1, count=4 * 8 * 131072, heads=8,
             dim=128, bits=3, dtype="float32"),
        # all 28 layers of Qwen2.5-1.5B at 4096 tokens decoded in one batched call for a bfloat16 attention
        dict(name="decode_layers_bf16", kind="decode", method="turboQuant", layers=28, count=2 * 4096, heads=2,
             dim=128, bits=4, dtype="bfloat16"),
        # one layer's per-channel keys, heads of 64, decoded to float16
        dict(name="decode_keys_kivi_f16", kind="decode_keys", heads=8, tokens=32768, dim=64, bits=4, group=64,
             dtype="float16"),
        # one query token of a Qwen2.5-1.5B layer over 2000 tokens, keys with the projection's bias removed
        dict(name="attend_bias_short", kind="attend", keys="bias", method="turboQuant", kv=2, queries=6, tokens=2000,
             dim=128, kbits=4, vbits=4, group=0),
        # one query token of a Llama-3-8B layer over 16000 tokens
        dict(name="attend_llama", kind="attend", keys="vector", method="turboQuant", kv=8, queries=4, tokens=16000,
             dim=128, kbits=4, vbits=4, group=0),
        # the long-context configuration: per-channel keys of four bits, values of three, 131072 tokens
        dict(name="attend_kivi_long", kind="attend", keys="channel", method="turboQuant", kv=8, queries=4,
             tokens=131072, dim=128, kbits=4, vbits=3, group=64),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["append", "append_keys", "encode", "encode", "encode", "encode_keys", "encode_keys", "decode",
                       "decode", "decode_keys", "attend", "attend", "attend", "attend"])
    bits = rng.choice([2, 3, 4, 4, 8])
    dtype = rng.choice(["float32", "float16", "bfloat16", "bfloat16"])
    method = rng.choice(["turboQuant", "turboQuant", "polarQuant"])
    heads = rng.choice([1, 2, 8, 12])
    if kind == "append":
        return dict(kind=kind, method=method, layers=rng.randint(4, 48), heads=heads, at=rng.randint(0, 2000),
                    dim=rng.choice([64, 128, 256]), bits=bits, dtype=dtype)
    if kind == "append_keys":
        return dict(kind=kind, heads=rng.choice([1, 2, 8]), tokens=_log(rng, 1, 20000),
                    dim=rng.choice([64, 80, 96, 128]), bits=bits, group=rng.choice([32, 64, 128]), dtype=dtype)
    if kind == "encode":
        tokens = max(1, _log(rng, 16, LAYER_VECTORS) // heads)
        return dict(kind=kind, method=method, count=tokens * heads, heads=heads, dim=rng.choice([64, 128, 128, 256]),
                    bits=bits, dtype=dtype)
    if kind in ("encode_keys", "decode_keys"):
        group = rng.choice([32, 64, 64, 128])
        tokens = max(1, _log(rng, 16, LAYER_VECTORS) // heads)
        if rng.random() < 0.5:
            tokens = max(group, tokens // group * group)
        return dict(kind=kind, heads=heads, tokens=tokens, dim=rng.choice([64, 80, 96, 128, 128]), bits=bits,
                    group=group, dtype=dtype)
    if kind == "decode":
        layers = rng.choice([1, 1, rng.randint(4, 48)])
        tokens = max(1, _log(rng, 16, LAYER_VECTORS // layers) // heads)
        return dict(kind=kind, method=method, layers=layers, count=tokens * heads, heads=heads,
                    dim=rng.choice([64, 128, 128, 256]), bits=bits, dtype=dtype)
    keys = rng.choice(["vector", "channel", "channel", "bias"])
    return dict(kind=kind, keys=keys, method=method, kv=rng.choice([1, 2, 4, 8, 12]), queries=rng.choice([1, 4, 4, 6, 8]),
                tokens=_log(rng, 64, 65536), dim=rng.choice([64, 128, 128]), kbits=rng.choice([2, 3, 4, 4]),
                vbits=rng.choice([2, 3, 4, 4]), group=rng.choice([64, 128]) if keys == "channel" else 0)


# ----------------------------------------------------------------------------------------- inputs
def _gen(seed: int):
    return torch.Generator(device="cuda").manual_seed(seed)


def _values(gen, tokens: int, heads: int, d: int, dtype: str):
    """Token-major heavy-tailed vectors, each head with a scale of its own, as a value cache holds them."""
    return W.gpt2_values(torch, gen, "cuda", tokens=tokens, heads=heads, d=d).to(DTYPES[dtype])


def _keys(gen, heads: int, tokens: int, d: int, dtype: str):
    """Head-major keys with uneven channels, outliers and a bias, as a key cache holds them."""
    return W.biased_keys(torch, gen, "cuda", heads, tokens, d).to(DTYPES[dtype])


def _encoded(q, x, cfg, key_bias=None):
    n = x.numel() // cfg.dim
    codes = torch.empty(n * cfg.codeStride, dtype=torch.uint8, device="cuda")
    scales = torch.empty(n, dtype=torch.float32, device="cuda")
    q.enqueueEncode(x, codes, scales, n, cfg, keyBias=key_bias)
    return codes, scales


def _key_calls(case, cfg):
    """(tokens, token offset, group offset) of each call over head-major keys."""
    heads, tokens = case["heads"], case["tokens"]
    if tokens % cfg.groupSize == 0:
        return [(heads * tokens, 0, 0)]
    return [(tokens, h * tokens, h * cfg.groupCount(tokens)) for h in range(heads)]


def _key_buffers(case, cfg):
    heads, tokens = case["heads"], case["tokens"]
    codes = torch.empty(heads * tokens * cfg.codeStride, dtype=torch.uint8, device="cuda")
    ranges = torch.empty(heads * cfg.groupCount(tokens) * 2 * cfg.dim, dtype=torch.float16, device="cuda")
    return codes, ranges


def _encode_keys(s):
    cfg, elem = s["cfg"], s["x"].element_size()
    for n, tok, grp in s["calls"]:
        s["q"].enqueuePerChannelEncode(s["x"], s["codes"], s["ranges"], n, cfg, inputOffset=tok * cfg.dim * elem,
                                       codesOffset=tok * cfg.codeStride, rangesOffset=grp * cfg.rangeStride)


def _rope(tokens: int, d: int):
    inv = 1.0 / 1e6 ** (torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)
    ang = torch.arange(tokens, dtype=torch.float64, device="cuda")[:, None] * inv[None, :]
    return tuple(torch.cat([t] * 2, 1).float().contiguous() for t in (torch.cos(ang), torch.sin(ang)))


def prepare(case: dict, seed: int) -> dict:
    q, gen, kind = P.PITCH(SEED), _gen(seed), case["kind"]
    s = {"kind": kind, "q": q}
    if kind == "append":
        cfg = q.config(case["method"], case["dim"], case["bits"])
        layers, heads, at = case["layers"], case["heads"], case["at"]
        x = torch.stack([_values(gen, 1, heads, cfg.dim, case["dtype"]) for _ in range(layers)])
        codes = torch.zeros((layers, (at + 1) * heads * cfg.codeStride), dtype=torch.uint8, device="cuda")
        scales = torch.zeros((layers, (at + 1) * heads), dtype=torch.float32, device="cuda")
        s.update(cfg=cfg, x=x, codes=codes, scales=scales, count=heads, at=at * heads,
                 table=P.EncodeBatch(q, cfg, list(x), list(codes), list(scales)))
    elif kind == "append_keys":
        cfg = q.channelConfig(case["dim"], case["bits"], case["group"])
        heads, tokens = case["heads"], case["tokens"]
        x = _keys(gen, heads, tokens, cfg.dim, case["dtype"])
        codes, ranges = _key_buffers(case, cfg)
        codes, ranges = codes.view(heads, -1), ranges.view(heads, -1)
        for h in range(heads):
            if tokens > 1:
                q.enqueuePerChannelEncode(x[h], codes[h], ranges[h], tokens - 1, cfg)
        s.update(cfg=cfg, x=x, codes=codes, ranges=ranges, heads=heads, tokens=tokens)
    elif kind == "encode":
        cfg = q.config(case["method"], case["dim"], case["bits"])
        n = case["count"]
        x = _values(gen, n // case["heads"], case["heads"], cfg.dim, case["dtype"])
        s.update(cfg=cfg, x=x, n=n, codes=torch.empty(n * cfg.codeStride, dtype=torch.uint8, device="cuda"),
                 scales=torch.empty(n, dtype=torch.float32, device="cuda"))
    elif kind in ("encode_keys", "decode_keys"):
        cfg = q.channelConfig(case["dim"], case["bits"], case["group"])
        x = _keys(gen, case["heads"], case["tokens"], cfg.dim, case["dtype"])
        codes, ranges = _key_buffers(case, cfg)
        s.update(cfg=cfg, x=x, codes=codes, ranges=ranges, calls=_key_calls(case, cfg))
        if kind == "decode_keys":
            _encode_keys(s)
            s.update(out=torch.empty_like(s.pop("x")))
    elif kind == "decode":
        cfg = q.config(case["method"], case["dim"], case["bits"])
        n, layers = case["count"], case["layers"]
        x = _values(gen, layers * n // case["heads"], case["heads"], cfg.dim, case["dtype"])
        codes, scales = _encoded(q, x, cfg)
        out = x.view(layers, -1).zero_()
        s.update(cfg=cfg, codes=codes, scales=scales, out=out, n=n, layers=layers)
        if layers > 1:
            s["table"] = P.DecodeBatch(q, cfg, list(codes.view(layers, -1)), list(scales.view(layers, -1)), list(out))
    else:
        kv, nq, T, d = case["kv"], case["queries"], case["tokens"], case["dim"]
        vcfg = q.config(case["method"], d, case["vbits"])
        out = torch.empty((kv, nq, d), device="cuda")
        lse = torch.empty((kv, nq), device="cuda")
        more = {}
        if case["keys"] == "channel":
            G = case["group"]
            kcfg = q.channelConfig(d, case["kbits"], G)
            stride = -(-T // G) * G    # head-major rows padded to whole groups, as the operator asks
            kc = torch.zeros(kv * stride * kcfg.codeStride, dtype=torch.uint8, device="cuda")
            ks = torch.zeros(kv * (stride // G) * 2 * d, dtype=torch.float16, device="cuda")
            x = _keys(gen, kv, T, d, "float32")
            for h in range(kv):
                q.enqueuePerChannelEncode(x[h], kc, ks, T, kcfg, codesOffset=h * stride * kcfg.codeStride,
                                          rangesOffset=h * (stride // G) * kcfg.rangeStride)
            vc = torch.zeros(kv * stride * vcfg.codeStride, dtype=torch.uint8, device="cuda")
            vs = torch.zeros(kv * stride, dtype=torch.float32, device="cuda")
            v = _values(gen, T, kv, d, "float32").transpose(0, 1).contiguous()
            for h in range(kv):
                q.enqueueEncode(v[h], vc, vs, T, vcfg, codesOffset=h * stride * vcfg.codeStride,
                                scalesOffset=h * stride * 4)
            query = torch.randn((kv, nq, d), generator=gen, device="cuda") * 0.3
            ws = P.attention_workspace_bytes(vcfg, vcfg, T, nq, kv)
        else:    # token-major caches, as appends of whole tokens write them
            kcfg = q.config(case["method"], d, case["kbits"])
            x = torch.randn((T, kv, d), generator=gen, device="cuda")
            if case["keys"] == "bias":
                cos, sin = _rope(T, d)
                b = torch.randn((kv, d), generator=gen, device="cuda") * 5
                more["keyBias"] = P.KeyBias(b, cos, sin, firstPosition=0, heads=kv)
                half = torch.cat([-b[:, d // 2:], b[:, :d // 2]], 1)
                x = (x + b * cos[:, None] + half * sin[:, None]).contiguous()
            kc, ks = _encoded(q, x, kcfg, more.get("keyBias"))
            vc, vs = _encoded(q, _values(gen, T, kv, d, "float32"), vcfg)
            more.update(tokenStride=kv, headStride=1)
            query = torch.randn((kv, nq, d), generator=gen, device="cuda") * (0.7 if "keyBias" in more else 2.0)
            ws = P.attention_workspace_bytes(kcfg, vcfg, T, nq, kv)
        s.update(kcfg=kcfg, vcfg=vcfg, query=query, kc=kc, ks=ks, vc=vc, vs=vs, out=out, lse=lse, more=more,
                 ws=torch.empty(ws, dtype=torch.uint8, device="cuda"), T=T, nq=nq, kv=kv)
    return s


def run(s: dict):
    q, kind = s["q"], s["kind"]
    if kind == "append":
        s["table"].enqueue(s["count"], codesOffsets=s["at"] * s["cfg"].codeStride, scalesOffsets=s["at"] * 4)
        return s["codes"], s["scales"]
    if kind == "append_keys":
        for h in range(s["heads"]):
            q.enqueuePerChannelAppend(s["x"][h], s["codes"][h], s["ranges"][h], s["tokens"], 1, s["cfg"])
        return s["codes"], s["ranges"]
    if kind == "encode":
        q.enqueueEncode(s["x"], s["codes"], s["scales"], s["n"], s["cfg"])
        return s["codes"], s["scales"]
    if kind == "encode_keys":
        _encode_keys(s)
        return s["codes"], s["ranges"]
    if kind == "decode":
        if s["layers"] > 1:
            s["table"].enqueue(s["n"])
        else:
            q.enqueueDecode(s["codes"], s["scales"], s["out"], s["n"], s["cfg"])
        return s["out"]
    if kind == "decode_keys":
        cfg, elem = s["cfg"], s["out"].element_size()
        for n, tok, grp in s["calls"]:
            q.enqueuePerChannelDecode(s["codes"], s["ranges"], s["out"], n, cfg, codesOffset=tok * cfg.codeStride,
                                      rangesOffset=grp * cfg.rangeStride, outputOffset=tok * cfg.dim * elem)
        return s["out"]
    q.enqueueAttentionDecode(s["query"], s["kc"], s["ks"], s["vc"], s["vs"], s["out"], s["T"], s["kcfg"], s["vcfg"],
                             qPerKv=s["nq"], kvHeads=s["kv"], lse=s["lse"], workspace=s["ws"], **s["more"])
    return s["out"], s["lse"]


# ----------------------------------------------------------------------------------------- what a pass cannot do without
def work(case: dict) -> dict:
    kind, d = case["kind"], case["dim"]
    elem = 4 if case.get("dtype", "float32") == "float32" else 2
    stride = P.code_stride_bytes
    rotate = d * math.log2(d)
    if kind in ("append", "encode", "decode"):
        n = case["layers"] * case["heads"] if kind == "append" else case.get("layers", 1) * case["count"]
        return {"bytes": n * (d * elem + stride(d, case["bits"]) + 4), "flops": n * (rotate + 4 * d)}
    if kind == "append_keys":
        n = case["heads"] * ((case["tokens"] - 1) % case["group"] + 1)
        return {"bytes": n * (d * elem + stride(d, case["bits"])) + case["heads"] * 4 * d, "flops": n * 5 * d}
    if kind in ("encode_keys", "decode_keys"):
        n, groups = case["heads"] * case["tokens"], case["heads"] * -(-case["tokens"] // case["group"])
        return {"bytes": n * (d * elem + stride(d, case["bits"])) + groups * 4 * d, "flops": n * 4 * d}
    T, kv, nq = case["tokens"], case["kv"], case["queries"]
    nbytes = kv * T * (stride(d, case["kbits"]) + stride(d, case["vbits"]) + 4) + kv * nq * d * 8
    nbytes += kv * -(-T // case["group"]) * 4 * d if case["keys"] == "channel" else kv * T * 4
    flops = 4 * kv * nq * T * d
    if case["keys"] == "bias":
        nbytes += T * d * 8
        flops += 4 * kv * nq * T * d
    return {"bytes": nbytes, "flops": flops}


# Tolerances, each about four times the largest difference seen between the library and exact(), over the range:
# codes and ranges are the reference's bits (a code may differ only at a tie); scales are float64 sums rounded once;
# float32 decodes carry the roundings of a float32 transform, and a 16-bit decode differs from the unrounded value by
# its own rounding (2^-9 of the value at most for bfloat16, 2^-12 for float16, a third of that in the 2-norm); the
# attention over per-channel keys with outlying channels errs by 5e-6 (large scores, rounded in float32, in exponents).
def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("append_keys", "encode_keys"):
        return {"rel": 5e-4, "max": 2e-3, "differ": 0.0}    # the ranges' float16 rounding against exact()
    if kind in ("append", "encode"):
        return {"rel": 3e-7, "max": 5e-7, "differ": 1e-6}
    if kind in ("decode", "decode_keys"):
        return {"float32": {"rel": 1e-6, "max": 1e-5}, "float16": {"rel": 8e-4, "max": 4e-3},
                "bfloat16": {"rel": 6e-3, "max": 3e-2}}[case["dtype"]]
    return {"rel": 2e-5, "max": 2e-4}


# ----------------------------------------------------------------------------------------- the same in 64 bits
def _signs(d: int):
    """+-1 of the rotation: the lowest bit of a PCG hash of seed + i."""
    out = []
    for i in range(d):
        state = ((SEED + i) * 747796405 + 2891336453) & 0xFFFFFFFF
        word = (((state >> ((state >> 28) + 4)) ^ state) * 277803737) & 0xFFFFFFFF
        out.append(1.0 if ((word >> 22) ^ word) & 1 else -1.0)
    return torch.tensor(out, dtype=torch.float64, device="cuda")


def _hadamard(x):
    n, d = x.shape
    h = 1
    while h < d:
        v = x.view(n, d // (2 * h), 2, h)
        x = torch.stack([v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]], 2).view(n, d)
        h *= 2
    return x / math.sqrt(d)


def _unpack(codes, n: int, d: int, b: int):
    w = codes.view(torch.int32).view(n, -1).to(torch.int64) & 0xFFFFFFFF
    pos = torch.arange(d, device="cuda") * b
    wi, sh = pos // 32, pos % 32
    lo = w[:, wi] >> sh
    hi = w[:, torch.clamp(wi + 1, max=w.shape[1] - 1)] << (32 - sh)
    return (lo | hi) & ((1 << b) - 1)


def _decoded(codes, scales, n: int, cfg):
    """The vectors that per-vector codes and scales stand for."""
    d, b = cfg.dim, cfg.bits
    c = _unpack(codes, n, d, b)
    if cfg.method.value == "turboQuant":
        path = Path(P.__file__).resolve().parent / "data" / "codebooks.json"
        book = torch.tensor(json.loads(path.read_text())["%d_%d" % (d, b)], dtype=torch.float32, device="cuda")
        y = book.double()[c]
    else:
        r, theta = c[:, 0::2] / (2 ** b - 1), c[:, 1::2] * (2 * math.pi / 2 ** b)
        y = torch.stack([r * torch.cos(theta), r * torch.sin(theta)], 2).view(n, d)
    return _hadamard(y) * _signs(d) * scales.double()[:, None]


def _decoded_keys(codes, ranges, n: int, cfg):
    d, G = cfg.dim, cfg.groupSize
    r = ranges.double().view(-1, 2, d)
    lo, step = r[:, 0], (r[:, 1] - r[:, 0]) / (2 ** cfg.bits - 1)
    step = torch.where(step == 0, torch.ones_like(step), step)
    g = torch.arange(n, device="cuda") // G
    return _unpack(codes, n, d, cfg.bits) * step[g] + lo[g]


def _scales(x, cfg):
    x = x.double().view(-1, cfg.dim)
    if cfg.method.value == "turboQuant":
        return x.norm(dim=1)
    y = _hadamard(x * _signs(cfg.dim))
    return torch.hypot(y[:, 0::2], y[:, 1::2]).amax(1)


def _ranges(x, heads: int, G: int):
    """[head][group][min row, max row] of head-major keys, unrounded."""
    x = x.double().view(heads, -1, x.shape[-1])
    parts = [torch.stack([x[:, i:i + G].amin(1), x[:, i:i + G].amax(1)], 1) for i in range(0, x.shape[1], G)]
    return torch.stack(parts, 1)


def exact(case: dict, seed: int):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "append":
        s["scales"][:, s["at"]:] = 0
        out = s["scales"].double()
        out[:, s["at"]:] = _scales(s["x"], s["cfg"]).view(out.shape[0], -1)
        return None, out
    if kind == "encode":
        return None, _scales(s["x"], s["cfg"])
    if kind in ("append_keys", "encode_keys"):
        r = _ranges(s["x"], case["heads"], case["group"])
        return None, r.reshape(s["ranges"].shape)
    if kind == "decode":
        n = s["n"] * s["layers"]
        return _decoded(s["codes"], s["scales"], n, s["cfg"]).view(s["out"].shape)
    if kind == "decode_keys":
        cfg, d = s["cfg"], s["cfg"].dim
        parts = [_decoded_keys(s["codes"][tok * cfg.codeStride:(tok + n) * cfg.codeStride],
                               s["ranges"][grp * 2 * d:(grp + cfg.groupCount(n)) * 2 * d], n, cfg)
                 for n, tok, grp in s["calls"]]
        return torch.cat(parts).view(s["out"].shape)
    kv, T, d = s["kv"], s["T"], case["dim"]
    rows = s["vs"].numel()
    V = _decoded(s["vc"], s["vs"], rows, s["vcfg"])
    if case["keys"] == "channel":
        K = _decoded_keys(s["kc"], s["ks"], rows, s["kcfg"]).view(kv, -1, d)[:, :T]
        V = V.view(kv, -1, d)[:, :T]
    else:
        K = _decoded(s["kc"], s["ks"], rows, s["kcfg"]).view(T, kv, d).transpose(0, 1)
        V = V.view(T, kv, d).transpose(0, 1)
        if case["keys"] == "bias":
            kb = s["more"]["keyBias"]
            b, cos, sin = kb.bias.double(), kb.cos.double(), kb.sin.double()
            half = torch.cat([-b[:, d // 2:], b[:, :d // 2]], 1)
            K = K + b[:, None] * cos + half[:, None] * sin
    scores = torch.stack([s["query"][h].double() @ K[h].contiguous().t() for h in range(kv)]) / math.sqrt(d)
    lse = torch.logsumexp(scores, -1)
    p = torch.exp(scores - lse[..., None])
    return torch.stack([p[h] @ V[h].contiguous() for h in range(kv)]), lse
