"""The 16-bit matrix-core attention kernels (pitch_attn_codes.hip) at the sizes where their tiling can go wrong: one
token, tiles of 64 tokens and their edges, one workgroup per KV head and the first sizes of several, chunks that end in
a partial tile, and one to eight query heads (two row layouts), for each kind of caches and a width on every table path.

Bar: 1e-5 relative L2 per query and 1e-5 on the log-sum-exp, as tests/test_gpu_attention.py derives it (float32
accumulation; the kernels' own operands hold 22 bits and more), and 1e-4 where scores reach 40 and more, as there. Values
of very uneven scales keep the bar too: a token's weight p n is held relative to the largest one of its tile of 64
tokens (per query head), in two float16 parts, of 22 bits down to 2^-28 of the largest and to 2^-49 of it at all.
"""
import math

import numpy as np
import pytest

from oracle import pitch_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _packed(rng, kv, rows, d, bits):
    codes = rng.integers(0, 2 ** bits, (kv, rows, d))
    return codes, np.frombuffer(b"".join(O.pack_codes(c, bits) for c in codes), np.uint8).reshape(kv, rows, -1)


def _compare(out, lse, ref_out, ref_lse, label, tol=TOL):
    for i in range(ref_out.shape[0]):
        e = np.linalg.norm(out[i] - ref_out[i]) / np.linalg.norm(ref_out[i])
        assert e < tol, f"{label}: query {i} relative L2 {e}"
    assert (np.abs(lse - ref_lse) / np.maximum(1.0, np.abs(ref_lse))).max() < tol, label


def _dev(q, *arrays):
    import torch
    return [torch.from_numpy(np.ascontiguousarray(a)).to(q.device) for a in arrays]


# unequal widths reach the kernels at every length, with one query only those below four bits (a call of 2 and 4 bits from
# 769 tokens to 32768 over all heads runs pitch_attention.hip's)
VECTOR = [("turboQuant", 4, 3, 128, 4, 2), ("turboQuant", 2, 4, 64, 1, 3), ("polarQuant", 3, 4, 128, 8, 1),
          ("turboQuant", 3, 2, 64, 5, 2), ("turboQuant", 2, 3, 64, 1, 3)]
TOKENS = [1, 63, 64, 65, 768, 769, 1023, 1024, 1025, 1153, 8191, 20001]


@pytest.mark.parametrize("tokens", TOKENS)
@pytest.mark.parametrize("method,kb,vb,d,nq,kv", VECTOR)
def test_vector_keys(q, method, kb, vb, d, nq, kv, tokens):
    """Token-major caches; the values' scales span nine powers of two."""
    import torch
    import pitch_amd as P
    label = f"{method} k{kb} v{vb} d={d} nq={nq} kv={kv} T={tokens}"
    print(label, flush=True)
    rng = np.random.default_rng(tokens + d + nq)
    kc, kp = _packed(rng, kv, tokens, d, kb)
    vc, vp = _packed(rng, kv, tokens, d, vb)
    ks = np.exp(rng.uniform(1.5, 3.0, (kv, tokens))).astype(np.float32)
    vs = np.exp2(rng.uniform(-4.0, 5.0, (kv, tokens))).astype(np.float32)
    Q = rng.standard_normal((kv, nq, d)).astype(np.float32)
    dq, dkc, dks, dvc, dvs = _dev(q, Q, kp.transpose(1, 0, 2), ks.T, vp.transpose(1, 0, 2), vs.T)
    out, lse = torch.empty(kv, nq, d, device=q.device), torch.empty(kv, nq, device=q.device)
    q.enqueueAttentionDecode(dq, dkc, dks, dvc, dvs, out, tokens, P.QuantConfig(method, d, kb, 101),
                             P.QuantConfig(method, d, vb, 202), qPerKv=nq, kvHeads=kv, tokenStride=kv, headStride=1, lse=lse)
    out, lse = out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)
    for h in range(kv):
        ro, rl = O.attention_decode(Q[h].astype(np.float64), kc[h], ks[h], vc[h], vs[h], method, kb, method, vb,
                                    1 / math.sqrt(d), 101, 202)
        _compare(out[h], lse[h], ro, rl, f"{label} head {h}")


@pytest.mark.parametrize("tokens", TOKENS)
@pytest.mark.parametrize("method,kb,vb,d,nq,kv,group",
                         [("turboQuant", 4, 3, 128, 4, 2, 64), ("turboQuant", 2, 2, 64, 8, 1, 128),
                          ("turboQuant", 3, 4, 128, 6, 1, 64), ("turboQuant", 3, 3, 64, 2, 3, 64),
                          ("polarQuant", 4, 4, 128, 4, 2, 64), ("polarQuant", 2, 4, 64, 8, 1, 64),
                          ("polarQuant", 3, 2, 64, 1, 2, 128), ("polarQuant", 4, 3, 128, 6, 1, 128)])
def test_channel_keys(q, method, kb, vb, d, nq, kv, group, tokens):
    """Head-major per-channel keys with uneven channels, and a partial last group; values of either method."""
    import torch
    import pitch_amd as P
    label = f"channel k{kb} {method} v{vb} d={d} nq={nq} kv={kv} G={group} T={tokens}"
    print(label, flush=True)
    rng = np.random.default_rng(tokens + d + nq + 7)
    stride = -(-tokens // group) * group
    K = (rng.standard_normal((kv, tokens, d)) * np.exp(rng.standard_normal((kv, 1, d))) + rng.standard_normal((kv, 1, d)))
    groups = stride // group
    kp = np.zeros((kv, stride, O.code_stride_bytes(d, kb)), np.uint8)
    kr = np.zeros((kv, groups, 2, d), np.float16)
    kcodes = []
    for h in range(kv):
        c, r = O.channel_encode(K[h].astype(np.float32), kb, group)
        kcodes.append(c)
        kp[h, :tokens] = np.frombuffer(O.pack_codes(c, kb), np.uint8).reshape(tokens, -1)
        kr[h] = r
    vc, vp = _packed(rng, kv, stride, d, vb)
    vs = np.exp(rng.uniform(-1.0, 1.0, (kv, stride))).astype(np.float32)
    Q = (0.5 * rng.standard_normal((kv, nq, d))).astype(np.float32)
    dq, dkp, dkr, dvp, dvs = _dev(q, Q, kp, kr, vp, vs)
    out, lse = torch.empty(kv, nq, d, device=q.device), torch.empty(kv, nq, device=q.device)
    q.enqueueAttentionDecode(dq, dkp, dkr, dvp, dvs, out, tokens, P.ChannelQuantConfig(d, kb, group),
                             P.QuantConfig(method, d, vb, 202), qPerKv=nq, kvHeads=kv, headStride=stride, lse=lse)
    out, lse = out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)
    for h in range(kv):
        Kd = O.channel_decode(kcodes[h], kr[h], kb, group).astype(np.float64)
        Vd = O.DECODERS[method](vc[h, :tokens], vs[h, :tokens].astype(np.float64), vb, 202)
        ro, rl = O.attend(Q[h].astype(np.float64), Kd, Vd, 1 / math.sqrt(d))
        _compare(out[h], lse[h], ro, rl, f"{label} head {h}")


# equal widths, whose keys and values share a table: lengths above those that attn_chunk serves
EQUAL = [("turboQuant", 4, 128, 4, 8, 5000), ("polarQuant", 3, 128, 8, 8, 5001), ("turboQuant", 4, 128, 1, 8, 8193),
         ("turboQuant", 2, 64, 2, 16, 9000), ("polarQuant", 4, 64, 8, 12, 12000), ("turboQuant", 3, 128, 3, 48, 1001)]


@pytest.mark.parametrize("head_major", [False, True])
@pytest.mark.parametrize("method,bits,d,nq,kv,tokens", EQUAL)
def test_equal_widths(q, method, bits, d, nq, kv, tokens, head_major):
    """Token-major caches put a chunk's heads on one XCD (8 chunks per head and more) or leave four chunks per head (48
    heads); head-major ones do neither. The first, a middle and the last head are compared."""
    import torch
    import pitch_amd as P
    print(f"{method} b={bits} d={d} nq={nq} kv={kv} T={tokens} head-major={head_major}", flush=True)
    rng = np.random.default_rng(tokens + d + nq)
    kc, kp = _packed(rng, kv, tokens, d, bits)
    vc, vp = _packed(rng, kv, tokens, d, bits)
    ks = np.exp(rng.uniform(1.5, 3.0, (kv, tokens))).astype(np.float32)
    vs = np.exp(rng.uniform(-1.0, 1.0, (kv, tokens))).astype(np.float32)
    Q = rng.standard_normal((kv, nq, d)).astype(np.float32)
    order = (0, 1) if head_major else (1, 0)
    dq, dkc, dvc = _dev(q, Q, kp.transpose(*order, 2), vp.transpose(*order, 2))
    dks, dvs = _dev(q, ks.transpose(order), vs.transpose(order))
    out, lse = torch.empty(kv, nq, d, device=q.device), torch.empty(kv, nq, device=q.device)
    layout = dict(headStride=tokens) if head_major else dict(tokenStride=kv, headStride=1)
    q.enqueueAttentionDecode(dq, dkc, dks, dvc, dvs, out, tokens, P.QuantConfig(method, d, bits, 101),
                             P.QuantConfig(method, d, bits, 202), qPerKv=nq, kvHeads=kv, lse=lse, **layout)
    out, lse = out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)
    for h in (0, kv // 2, kv - 1):
        ro, rl = O.attention_decode(Q[h].astype(np.float64), kc[h], ks[h], vc[h], vs[h], method, bits, method, bits,
                                    1 / math.sqrt(d), 101, 202)
        _compare(out[h], lse[h], ro, rl, f"head {h}")


@pytest.mark.parametrize("nq", [4, 8])
@pytest.mark.parametrize("keys", ["equal", "unequal", "bias", "channel"])
def test_late_maxima(q, keys, nq):
    """Scores up to 40 and more whose size grows with the position, so that the maximum of every wave's second and later
    tiles is above that of the tiles before and its accumulators are rescaled: 24 KV heads of 250 tiles, 8 workgroups per
    head, two tiles per wave (four to six with eight queries or the key-bias term)."""
    import torch
    import pitch_amd as P
    print(keys, nq, flush=True)
    kv, tokens, d, vb, group = 24, 16000, 64, 4 if keys == "equal" else 3, 64
    rng = np.random.default_rng(nq)
    ramp = np.linspace(0.2, 1.0, tokens)
    vc, vp = _packed(rng, kv, tokens, d, vb)
    vs = np.exp(rng.uniform(-1.0, 1.0, (kv, tokens))).astype(np.float32)
    Q = rng.standard_normal((kv, nq, d)).astype(np.float32)
    more, heads = {}, (0, kv - 1)
    if keys == "channel":
        K = rng.standard_normal((kv, tokens, d)).astype(np.float32) * (10 * ramp[:, None]).astype(np.float32)
        enc = [O.channel_encode(K[h], 4, group) for h in range(kv)]
        kp = np.stack([np.frombuffer(O.pack_codes(c, 4), np.uint8).reshape(tokens, -1) for c, _ in enc])
        ks = np.stack([r for _, r in enc])
        kcfg = P.ChannelQuantConfig(d, 4, group)
        Kd = {h: O.channel_decode(*enc[h], 4, group).astype(np.float64) for h in heads}
    else:
        kc, kp = _packed(rng, kv, tokens, d, 4)
        ks = (80 * ramp * np.ones((kv, 1))).astype(np.float32)
        kcfg = P.QuantConfig("turboQuant", d, 4, 101)
        Kd = {h: O.turbo_decode(kc[h], ks[h].astype(np.float64), 4, 101) for h in heads}
        if keys == "bias":
            ang = np.arange(tokens)[:, None] * (1e4 ** -(np.arange(d // 2) / (d // 2)))[None]
            cos, sin = (np.concatenate([f(ang)] * 2, 1).astype(np.float32) for f in (np.cos, np.sin))
            b = rng.standard_normal((kv, d)).astype(np.float32)
            more["keyBias"] = P.KeyBias(*_dev(q, b, cos, sin), firstPosition=0, heads=kv)
            kp, ks, vp = kp.transpose(1, 0, 2), ks.T, vp.transpose(1, 0, 2)
            more.update(tokenStride=kv, headStride=1)
            for h in heads:
                half = np.concatenate([-b[h, d // 2:], b[h, :d // 2]])
                Kd[h] = Kd[h] + b[h].astype(np.float64) * cos + half.astype(np.float64) * sin
    dq, dkc, dks, dvc, dvs = _dev(q, Q, kp, ks, vp, vs.T if keys == "bias" else vs)
    out, lse = torch.empty(kv, nq, d, device=q.device), torch.empty(kv, nq, device=q.device)
    q.enqueueAttentionDecode(dq, dkc, dks, dvc, dvs, out, tokens, kcfg, P.QuantConfig("turboQuant", d, vb, 202),
                             qPerKv=nq, kvHeads=kv, lse=lse, **(more or dict(headStride=tokens)))
    out, lse = out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)
    for h in heads:
        Vd = O.turbo_decode(vc[h], vs[h].astype(np.float64), vb, 202)
        ro, rl = O.attend(Q[h].astype(np.float64), Kd[h], Vd, 1 / math.sqrt(d))
        assert rl.max() > 30, rl
        _compare(out[h], lse[h], ro, rl, f"{keys} head {h}", 1e-4)


@pytest.mark.parametrize("tokens", [1, 64, 65, 257, 4097])
@pytest.mark.parametrize("method,kb,vb,d,nq,kv", [("turboQuant", 4, 4, 128, 6, 2), ("polarQuant", 3, 2, 64, 2, 3)])
def test_key_bias(q, method, kb, vb, d, nq, kv, tokens):
    import torch
    import pitch_amd as P
    label = f"bias {method} k{kb} v{vb} d={d} nq={nq} kv={kv} T={tokens}"
    print(label, flush=True)
    rng = np.random.default_rng(tokens + d + nq + 11)
    first = 5
    kc, kp = _packed(rng, kv, tokens, d, kb)
    vc, vp = _packed(rng, kv, tokens, d, vb)
    ks = np.exp(rng.uniform(1.5, 2.5, (kv, tokens))).astype(np.float32)
    vs = np.exp(rng.uniform(-1.0, 1.0, (kv, tokens))).astype(np.float32)
    ang = np.arange(first + tokens)[:, None] * (1e4 ** -(np.arange(d // 2) / (d // 2)))[None]
    cos = np.concatenate([np.cos(ang)] * 2, 1).astype(np.float32)
    sin = np.concatenate([np.sin(ang)] * 2, 1).astype(np.float32)
    b = (3 * rng.standard_normal((kv, d))).astype(np.float32)
    Q = (0.4 * rng.standard_normal((kv, nq, d))).astype(np.float32)
    dq, dkc, dks, dvc, dvs, db, dcos, dsin = _dev(q, Q, kp.transpose(1, 0, 2), ks.T, vp.transpose(1, 0, 2), vs.T, b, cos, sin)
    out, lse = torch.empty(kv, nq, d, device=q.device), torch.empty(kv, nq, device=q.device)
    q.enqueueAttentionDecode(dq, dkc, dks, dvc, dvs, out, tokens, P.QuantConfig(method, d, kb, 101),
                             P.QuantConfig(method, d, vb, 202), qPerKv=nq, kvHeads=kv, tokenStride=kv, headStride=1,
                             lse=lse, keyBias=P.KeyBias(db, dcos, dsin, firstPosition=first, heads=kv))
    out, lse = out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)
    off = O.key_bias_offsets(b, cos, sin, first, tokens * kv, kv).reshape(tokens, kv, d).astype(np.float64)
    for h in range(kv):
        Kd = O.DECODERS[method](kc[h], ks[h].astype(np.float64), kb, 101) + off[:, h]
        Vd = O.DECODERS[method](vc[h], vs[h].astype(np.float64), vb, 202)
        ro, rl = O.attend(Q[h].astype(np.float64), Kd, Vd, 1 / math.sqrt(d))
        _compare(out[h], lse[h], ro, rl, f"{label} head {h}")


@pytest.mark.parametrize("tokens", [150, 3000, 20001])
@pytest.mark.parametrize("d,nq", [(128, 4), (64, 8)])
@pytest.mark.parametrize("what", ["huge scale without weight", "weight without scale", "wide scales", "tiny scales"])
def test_range_of_weights(q, what, d, nq, tokens):
    """A token's share of the output is p n, softmax weight times value scale. One token (the fourth, in a wave's first
    tile) has a value scale 2^60 times the others' and p = e^-70, or p near 1 and a zero value (an attention sink); or
    all scales span 2^-40 to 2^40, or lie near 2^-115. In float32 none of that costs precision."""
    import torch
    import pitch_amd as P
    print(what, d, nq, tokens, flush=True)
    rng = np.random.default_rng(tokens + d)
    kc, kp = _packed(rng, 1, tokens, d, 4)
    vc, vp = _packed(rng, 1, tokens, d, 3)
    ks = np.exp(rng.uniform(0.0, 1.0, (1, tokens))).astype(np.float32)
    vs = np.exp(rng.uniform(-1.0, 1.0, (1, tokens))).astype(np.float32)
    Q = rng.standard_normal((1, nq, d))
    k3 = O.turbo_decode(kc[0, 3:4], ks[0, 3:4].astype(np.float64), 4, 101)[0]
    score = {"huge scale without weight": -60.0, "weight without scale": 45.0}.get(what)
    if score is not None:    # the fourth token's score
        Q[0] += np.outer(score * math.sqrt(d) - Q[0] @ k3, k3 / (k3 @ k3))
    if what == "huge scale without weight":
        vs[0, 3] = 2.0 ** 60
    elif what == "weight without scale":
        vs[0, 3] = 0.0
    elif what == "wide scales":
        vs = np.exp2(rng.uniform(-40.0, 40.0, (1, tokens))).astype(np.float32)
    else:
        vs = np.exp2(rng.uniform(-116.0, -114.0, (1, tokens))).astype(np.float32)
    Q = Q.astype(np.float32)
    dq, dkc, dks, dvc, dvs = _dev(q, Q, kp, ks, vp, vs)
    out, lse = torch.empty(1, nq, d, device=q.device), torch.empty(1, nq, device=q.device)
    q.enqueueAttentionDecode(dq, dkc, dks, dvc, dvs, out, tokens, P.QuantConfig("turboQuant", d, 4, 101),
                             P.QuantConfig("turboQuant", d, 3, 202), qPerKv=nq, lse=lse)
    out, lse = out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)
    ro, rl = O.attention_decode(Q[0].astype(np.float64), kc[0], ks[0], vc[0], vs[0], "turboQuant", 4, "turboQuant", 3,
                                1 / math.sqrt(d), 101, 202)
    _compare(out[0], lse[0], ro, rl, f"{what} d={d} nq={nq} T={tokens}", TOL if score is None else 1e-4)


@pytest.mark.parametrize("tokens", [64, 65, 129, 1100, 2113])
@pytest.mark.parametrize("d,nq", [(128, 4), (64, 8)])
def test_infinities_and_nan(q, d, nq, tokens):
    """Two KV heads; the first head's last token, alone in its tile or not, has a key scale of infinity: a score of minus
    infinity takes no part (the queries come in pairs q and -q: one of each pair has it), plus infinity and a NaN scale
    give NaN, and an infinite value scale nothing finite. The second head does not notice."""
    import torch
    import pitch_amd as P
    print(d, nq, tokens, flush=True)
    rng = np.random.default_rng(tokens + d)
    kc, kp = _packed(rng, 2, tokens, d, 4)
    vc, vp = _packed(rng, 2, tokens, d, 3)
    ks, vs = (np.exp(rng.uniform(0.0, 1.0, (2, tokens))).astype(np.float32) for _ in range(2))
    Q = rng.standard_normal((2, nq // 2, d))
    Q = np.concatenate([Q, -Q], 1).astype(np.float32)
    last = O.turbo_decode(kc[0, -1:], np.ones(1), 4, 101)[0]
    plus = Q[0].astype(np.float64) @ last > 0

    def run(key, value):
        k, v = ks.copy(), vs.copy()
        k[0, -1] *= key
        v[0, -1] *= value
        dq, dkc, dks, dvc, dvs = _dev(q, Q, kp, k, vp, v)
        out, lse = torch.empty(2, nq, d, device=q.device), torch.empty(2, nq, device=q.device)
        q.enqueueAttentionDecode(dq, dkc, dks, dvc, dvs, out, tokens, P.QuantConfig("turboQuant", d, 4, 101),
                                 P.QuantConfig("turboQuant", d, 3, 202), qPerKv=nq, kvHeads=2, lse=lse)
        return out.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64)

    def reference(h, n):
        return O.attention_decode(Q[h].astype(np.float64), kc[h, :n], ks[h, :n], vc[h, :n], vs[h, :n], "turboQuant", 4,
                                  "turboQuant", 3, 1 / math.sqrt(d), 101, 202)

    inf, nan = float("inf"), float("nan")
    for key, value in ((inf, 1.0), (nan, 1.0), (1.0, inf), (1.0, nan)):
        out, lse = run(key, value)
        _compare(out[1], lse[1], *reference(1, tokens), f"head 1 beside {key} {value}")
        if key == inf:
            ro, rl = reference(0, tokens - 1)
            _compare(out[0][~plus], lse[0][~plus], ro[~plus], rl[~plus], "minus infinity")
            assert np.isnan(out[0][plus]).all()
        else:
            assert not np.isfinite(out[0]).any()


def test_threads_of_different_lengths(q):
    """Calls of one kernel variant from several threads, each on a stream of its own, with lengths that take four waves
    a workgroup and sixteen (different amounts of LDS): none is refused and each writes what it writes alone."""
    import threading

    import torch
    import pitch_amd as P
    d, nq, kv = 128, 4, 2
    rng = np.random.default_rng(5)
    kcfg, vcfg = P.QuantConfig("turboQuant", d, 4, 101), P.QuantConfig("turboQuant", d, 3, 202)

    def call(tokens):
        _, kp = _packed(rng, kv, tokens, d, 4)
        _, vp = _packed(rng, kv, tokens, d, 3)
        ks, vs = (np.exp(rng.uniform(0.0, 1.0, (kv, tokens))).astype(np.float32) for _ in range(2))
        args = _dev(q, rng.standard_normal((kv, nq, d)).astype(np.float32), kp, ks, vp, vs)
        ws = torch.empty(P.attention_workspace_bytes(kcfg, vcfg, tokens, nq, kv), dtype=torch.uint8, device=q.device)

        def run(out, stream=None):
            q.enqueueAttentionDecode(*args, out, tokens, kcfg, vcfg, qPerKv=nq, kvHeads=kv, workspace=ws, stream=stream)
        alone = torch.empty(kv, nq, d, device=q.device)
        run(alone)
        return run, alone

    calls = [call(t) for t in (200, 1024, 100, 900)]
    torch.cuda.synchronize()
    failed = []

    def work(run, alone):
        try:
            stream = torch.cuda.Stream()
            outs = [torch.full_like(alone, float("nan")) for _ in range(8)]
            torch.cuda.synchronize()
            for i in range(400):
                run(outs[i % 8], stream)
            stream.synchronize()
            assert all(torch.equal(o, alone) for o in outs)
        except Exception as e:  # noqa: BLE001 (reported by the main thread)
            failed.append(repr(e))

    threads = [threading.Thread(target=work, args=c) for c in calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
