"""The work split of the 16-bit matrix-core attention kernels (codes_split in pitch_attention.hip) against the
workspace that pitch_attention_workspace_size promises its callers: restated here, since a launch needs a GPU."""
import ctypes

import pytest

from pitch_amd import _lib


def codes_chunks(tokens: int, kv: int, bias: bool, cus: int) -> int:
    tiles = -(-tokens // 64)
    chunks = 1
    if tiles > (4 if bias else 16):
        chunks = cus // kv
        if chunks >= 8:
            chunks = chunks // 8 * 8
        most = tiles if bias else -(-tiles // 2)
        chunks = min(chunks, most) if chunks > most else min(max(chunks, 1), 128)
    per = -(-tiles // chunks)
    return -(-tiles // per)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dim", [64, 128])
def test_partials_fit_the_workspace(dim, bias):
    if not _lib.LIB_PATH.exists():
        pytest.skip("HIP library not built")
    lib = _lib.load()
    cfg = _lib.PitchConfigC(0, dim, 4, 1)
    out = ctypes.c_uint64()
    edges = {2 ** k + e for k in range(5, 22) for e in (-1, 0, 1, 63, 64, 65)} | set(range(1, 1400, 7))
    for cus in (1, 64, 256, 304):
        for kv in (1, 2, 3, 8, 12, 200):
            for tokens in sorted(edges):
                desc = _lib.PitchAttentionDescC(1, kv, tokens, 1, tokens, 1.0, 0)
                assert lib.pitch_attention_workspace_size(ctypes.byref(cfg), ctypes.byref(cfg), ctypes.byref(desc),
                                                          ctypes.byref(out)) == 0
                chunks = codes_chunks(tokens, kv, bias, cus)
                if chunks > 1:    # a single chunk writes the output itself
                    assert 4 * kv * chunks * (2 + dim) <= out.value, (cus, kv, tokens, chunks)
