"""16-bit vectors at d = 256, 512 and 1024 through the LDS-transposed encoder: codes and scales equal those of the
float32 entry point on the widened values, byte for byte, at counts around its wave and workgroup sizes (8, 4 and 2
vectors a wave, four waves) and over several rounds, from an input that is only 4-byte aligned, single and batched."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("method", ["turboQuant", "polarQuant"])
@pytest.mark.parametrize("dim,bits", [(256, 2), (256, 5), (512, 3), (512, 8), (1024, 4), (1024, 7)])
def test_equals_widened(q, dim, bits, method, dtype):
    import torch
    cfg = q.config(method, dim, bits)
    vpb = 4 * 2048 // dim
    gen = torch.Generator(device=q.device).manual_seed(dim + bits)
    total = 40 * 256 * vpb + 3
    x = torch.randn(total * dim + 2, generator=gen, device=q.device).to(getattr(torch, dtype))
    x[2 + 5 * dim:2 + 6 * dim] = 0                       # a zero vector
    wide = x[2:].float()
    codes, ref_codes = (torch.zeros(total * cfg.codeStride, dtype=torch.uint8, device=q.device) for _ in range(2))
    scales, ref_scales = (torch.zeros(total, device=q.device) for _ in range(2))
    for count in (1, vpb // 4 + 1, vpb - 1, vpb, vpb + 1, total):
        print(f"{method} {dtype} d={dim} b={bits} count={count}", flush=True)
        for t in (codes, ref_codes, scales, ref_scales):
            t.zero_()
        q.enqueueEncode(x, codes, scales, count, cfg, inputOffset=4)
        q.enqueueEncode(wide, ref_codes, ref_scales, count, cfg)
        assert torch.equal(codes, ref_codes) and torch.equal(scales, ref_scales)
    a, b, s = 3, vpb + 2, cfg.codeStride
    codes.zero_(), scales.zero_()
    q.enqueueEncodeBatch([(x, codes, scales, a, 4, 0, 0), (x, codes, scales, b, 4 + 2 * a * dim, a * s, 4 * a)], cfg)
    ref_codes[(a + b) * s:] = 0
    ref_scales[a + b:] = 0
    assert torch.equal(codes, ref_codes) and torch.equal(scales, ref_scales)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("dim,bits", [(256, 6), (512, 7), (1024, 8)])
def test_polar_sizes_of_both_encoders(q, dim, bits, dtype):
    """PolarQuant of 6 bits and more: calls of up to 2^12 coordinates and from 2^22 (eight bits: above it) run the
    transposed encoder, those between the team encoder, and so do the segments of a batch of as many; the same bytes on each side."""
    import torch
    cfg = q.config("polarQuant", dim, bits)
    gen = torch.Generator(device=q.device).manual_seed(dim + bits)
    total = (1 << 22) // dim + 1
    x = torch.randn(total * dim, generator=gen, device=q.device).to(getattr(torch, dtype))
    wide = x.float()
    s = cfg.codeStride
    ref_codes, ref_scales = torch.zeros(total * s, dtype=torch.uint8, device=q.device), torch.zeros(total, device=q.device)
    q.enqueueEncode(wide, ref_codes, ref_scales, total, cfg)
    for count in ((1 << 12) // dim, (1 << 12) // dim + 1, total - 2, total - 1, total):
        for batched in (False, True):
            print(f"{dtype} d={dim} b={bits} count={count} batched={batched}", flush=True)
            codes, scales = torch.zeros_like(ref_codes), torch.zeros_like(ref_scales)
            a = count // 3 if batched else 0
            if batched:
                q.enqueueEncodeBatch([(x, codes, scales, a, 0, 0, 0), (x, codes, scales, count - a, 2 * a * dim, a * s, 4 * a)],
                                     cfg)
            else:
                q.enqueueEncode(x, codes, scales, count, cfg)
            assert torch.equal(codes[:count * s], ref_codes[:count * s]) and not codes[count * s:].any()
            assert torch.equal(scales[:count], ref_scales[:count]) and not scales[count:].any()
