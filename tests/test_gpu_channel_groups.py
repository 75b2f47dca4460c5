"""Per-channel encode and decode at the group sizes where the wave kernels change: 32, 64 and 128 rows for the encoder,
32- and 64-token chunks for the decoder, and the sizes around them, with whole, partial and single-token last groups.
Codes, ranges and decoded values are the oracle's bits (zero extremes of both signs included)."""
import numpy as np
import pytest

from oracle import pitch_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("io", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("group", [1, 17, 31, 32, 33, 63, 65, 96, 100, 127, 128, 129, 160])
@pytest.mark.parametrize("dim,bits", [(64, 4), (80, 3), (96, 2), (128, 8), (36, 5)])
def test_bits(q, dim, bits, group, io):
    import torch
    print(f"d={dim} b={bits} G={group} {io}", flush=True)
    rng = np.random.default_rng(dim * 1000 + group)
    tokens = 3 * group + (group + 1) // 2
    x = rng.standard_normal((tokens, dim)).astype(np.float32) * np.exp(rng.standard_normal(dim)).astype(np.float32)
    x[:, 3] = np.abs(x[:, 3])
    x[rng.random(tokens) < 0.3, 3] = -0.0
    x[rng.random(tokens) < 0.3, 3] = 0.0        # a minimum of either zero
    t = torch.from_numpy(x).to(getattr(torch, io))
    wide = t.float().numpy()
    codes, ranges = O.channel_encode(wide, bits, group)
    cfg = q.channelConfig(dim, bits, group)
    dev = t.to(q.device)
    c = torch.zeros(tokens * cfg.codeStride, dtype=torch.uint8, device=q.device)
    r = torch.zeros(ranges.size, dtype=torch.int16, device=q.device)
    q.enqueuePerChannelEncode(dev, c, r, tokens, cfg)
    assert c.cpu().numpy().tobytes() == O.pack_codes(codes, bits)
    assert np.array_equal(r.cpu().numpy().view(np.uint16), ranges.reshape(-1).view(np.uint16))
    out = torch.zeros((tokens, dim), dtype=t.dtype, device=q.device)
    q.enqueuePerChannelDecode(c, r, out, tokens, cfg)
    want = O.to_io_bits(O.channel_decode(codes, ranges, bits, group), io)
    assert np.array_equal(out.cpu().view(torch.int32 if io == "float32" else torch.int16).numpy().view(want.dtype), want)


@pytest.mark.parametrize("io", ["float32", "bfloat16"])
@pytest.mark.parametrize("tokens", [130, 1000, 32768, 32769])
@pytest.mark.parametrize("group", [65, 96, 128])
@pytest.mark.parametrize("dim,bits", [(12, 2), (16, 8), (12, 5), (28, 4), (36, 3), (44, 3), (52, 2), (56, 6), (60, 5), (60, 8)])
def test_partial_slabs(q, dim, bits, group, tokens, io):
    """Groups of 65 to 128 rows whose channels do not fill slabs of 32: both encoders at both sides of their rule."""
    import torch
    print(f"d={dim} b={bits} G={group} {io} {tokens}", flush=True)
    rng = np.random.default_rng(dim * 1000 + group + tokens)
    x = rng.standard_normal((tokens, dim)).astype(np.float32)
    t = torch.from_numpy(x).to(getattr(torch, io))
    codes, ranges = O.channel_encode(t.float().numpy(), bits, group)
    cfg = q.channelConfig(dim, bits, group)
    c = torch.zeros(tokens * cfg.codeStride, dtype=torch.uint8, device=q.device)
    r = torch.zeros(ranges.size, dtype=torch.int16, device=q.device)
    q.enqueuePerChannelEncode(t.to(q.device), c, r, tokens, cfg)
    assert c.cpu().numpy().tobytes() == O.pack_codes(codes, bits)
    assert np.array_equal(r.cpu().numpy().view(np.uint16), ranges.reshape(-1).view(np.uint16))


@pytest.mark.parametrize("io", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("tokens", [1, 31, 32, 33, 64])
@pytest.mark.parametrize("dim,bits", [(64, 4), (80, 3), (84, 2), (128, 8)])
def test_decode_of_few_groups_of_32(q, dim, bits, tokens, io):
    """One group of 32 tokens, whole or not, and two: the decoders at both sides of their rule."""
    import torch
    print(f"d={dim} b={bits} {io} {tokens}", flush=True)
    rng = np.random.default_rng(dim + tokens)
    codes, ranges = O.channel_encode(rng.standard_normal((tokens, dim)).astype(np.float32), bits, 32)
    cfg = q.channelConfig(dim, bits, 32)
    c = torch.from_numpy(np.frombuffer(O.pack_codes(codes, bits), np.uint8).copy()).to(q.device)
    r = torch.from_numpy(ranges.reshape(-1).view(np.int16).copy()).to(q.device)
    out = torch.zeros((tokens, dim), dtype=getattr(torch, io), device=q.device)
    q.enqueuePerChannelDecode(c, r, out, tokens, cfg)
    want = O.to_io_bits(O.channel_decode(codes, ranges, bits, 32), io)
    assert np.array_equal(out.cpu().view(torch.int32 if io == "float32" else torch.int16).numpy().view(want.dtype), want)


@pytest.mark.parametrize("tokens", [4095, 4096, 4097, 5000])
@pytest.mark.parametrize("dim,bits,group", [(64, 3, 32), (80, 5, 16), (96, 6, 17), (128, 7, 32)])
def test_rows_of_small_groups(q, dim, bits, group, tokens):
    """float32 groups of up to 32 rows, widths that are packed code by code: 64 and 32 rows per wave."""
    import torch
    print(f"d={dim} b={bits} G={group} {tokens}", flush=True)
    x = np.random.default_rng(dim + tokens).standard_normal((tokens, dim)).astype(np.float32)
    codes, ranges = O.channel_encode(x, bits, group)
    cfg = q.channelConfig(dim, bits, group)
    c = torch.zeros(tokens * cfg.codeStride, dtype=torch.uint8, device=q.device)
    r = torch.zeros(ranges.size, dtype=torch.int16, device=q.device)
    q.enqueuePerChannelEncode(torch.from_numpy(x).to(q.device), c, r, tokens, cfg)
    assert c.cpu().numpy().tobytes() == O.pack_codes(codes, bits)
    assert np.array_equal(r.cpu().numpy().view(np.uint16), ranges.reshape(-1).view(np.uint16))


@pytest.mark.parametrize("io", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows", [1, 31, 32, 33, 64, 65, 127])
@pytest.mark.parametrize("dim,bits,group", [(64, 4, 128), (80, 3, 128), (128, 8, 100), (28, 5, 65), (128, 2, 64)])
def test_appends_to_a_short_last_group(q, dim, bits, group, rows, io):
    """Appends of single tokens to the last of two groups: what is written equals one encode of all tokens, for every count
    of rows that the last group can have, and the first group stays."""
    import torch
    rows = min(rows, group)
    print(f"d={dim} b={bits} G={group} rows={rows} {io}", flush=True)
    tokens = group + rows
    x = np.random.default_rng(dim + rows).standard_normal((tokens, dim)).astype(np.float32)
    t = torch.from_numpy(x).to(getattr(torch, io))
    codes, ranges = O.channel_encode(t.float().numpy(), bits, group)
    cfg = q.channelConfig(dim, bits, group)
    dev = t.to(q.device)
    c = torch.zeros(tokens * cfg.codeStride, dtype=torch.uint8, device=q.device)
    r = torch.zeros(ranges.size, dtype=torch.int16, device=q.device)
    q.enqueuePerChannelEncode(dev, c, r, tokens - 1, cfg)
    q.enqueuePerChannelAppend(dev, c, r, tokens, 1, cfg)
    assert c.cpu().numpy().tobytes() == O.pack_codes(codes, bits)
    assert np.array_equal(r.cpu().numpy().view(np.uint16), ranges.reshape(-1).view(np.uint16))
