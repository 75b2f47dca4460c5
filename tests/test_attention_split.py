"""The work split of the 16-bit matrix-core attention kernels, as the library computes it for a launch
(pitch_selftest_attention_split): every chunk's partial results fit the workspace that callers are told to bring, on
devices of any size and for a workspace sized with any chunk length, and the split covers the tokens."""
import ctypes

import pytest

from pitch_amd import _lib

EDGES = sorted({2 ** k + e for k in range(5, 22) for e in (-1, 0, 1, 63, 64, 65)} | set(range(1, 1400, 7))
               | {2 ** 32 - 1, 2 ** 32, 2 ** 36})


@pytest.fixture(scope="module")
def split(built_library):
    lib = _lib.load()
    out = (ctypes.c_uint64 * 4)()

    def call(dim, tokens, kv, bias, cus, ws_chunk=0, head_major=0):
        assert lib.pitch_selftest_attention_split(dim, tokens, kv, bias, head_major, cus, ws_chunk, out) == 0
        return tuple(out)
    return call


@pytest.mark.parametrize("ws_chunk", [0, 64, 128, 1024])
@pytest.mark.parametrize("bias,head_major", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("dim", [64, 128])
def test_partials_fit_the_workspace(split, dim, bias, head_major, ws_chunk):
    for cus in (1, 64, 256, 304, 1024):
        for kv in (1, 2, 3, 8, 12, 48, 129, 200, 300, 65535):
            for tokens in EDGES:
                chunk, chunks, waves, floats = split(dim, tokens, kv, bias, cus, ws_chunk, head_major)
                label = (cus, kv, tokens, chunk, chunks)
                assert chunk % 64 == 0 and chunk < 2 ** 31 and (chunks - 1) * chunk < tokens <= chunks * chunk, label
                assert chunks <= 128 and 4 <= waves <= 16, label
                if chunks > 1:    # a single chunk writes the output itself
                    assert kv * chunks * (2 + dim) <= floats, label


def test_token_major_chunks_stay_on_few_xcds(split):
    """Five chunks per head would spread the rows of one token over all XCDs; head-major caches and calls with the key-bias
    term keep all they can have."""
    for kv in (43, 48, 51):
        assert split(128, 200000, kv, 0, 256)[1] == 4
        assert split(128, 200000, kv, 0, 256, head_major=1)[1] == split(128, 200000, kv, 1, 256)[1] == 5


# (dim, tokens, KV heads, queries, key bits, value bits, head-major): whether attention over per-vector caches runs the
# 16-bit matrix-core kernels on 256 compute units, as it measured faster; both sides of each line of the rule.
ROUTES = [
    (128, 300, 8, 4, 4, 4, 0, 1), (64, 512, 1, 1, 2, 2, 1, 1), (64, 513, 1, 1, 2, 2, 1, 0),
    (64, 768, 2, 1, 4, 3, 0, 1), (128, 4096, 8, 4, 4, 4, 0, 0), (128, 4097, 8, 4, 4, 4, 0, 1),
    (64, 131072, 1, 4, 3, 3, 0, 0), (64, 131073, 1, 4, 3, 3, 0, 1), (128, 4096, 16, 1, 4, 4, 0, 0),
    (128, 4097, 12, 1, 4, 4, 0, 1), (128, 4096, 16, 1, 3, 3, 0, 1), (128, 2000, 24, 1, 4, 4, 0, 0),
    (128, 16000, 2, 1, 4, 3, 0, 0), (128, 16000, 2, 1, 3, 2, 0, 1), (128, 16000, 2, 2, 4, 3, 0, 1),
    (64, 20000, 2, 1, 2, 4, 0, 1), (64, 8000, 20, 1, 4, 4, 0, 0), (64, 8000, 20, 2, 4, 4, 0, 1),
    (64, 16000, 16, 1, 4, 4, 0, 1), (64, 32000, 12, 1, 4, 4, 0, 1), (64, 65536, 12, 1, 4, 4, 0, 0),
    (64, 65536, 12, 4, 4, 4, 0, 1), (128, 8000, 20, 1, 2, 2, 0, 0), (128, 8000, 20, 1, 3, 3, 0, 1),
    (128, 8000, 28, 1, 2, 2, 0, 1), (64, 8000, 40, 1, 4, 4, 0, 0), (64, 8000, 40, 4, 4, 4, 0, 0),
    (64, 8000, 40, 4, 2, 2, 0, 1), (64, 8000, 40, 8, 4, 4, 0, 1), (64, 8000, 36, 4, 2, 2, 0, 0),
    (64, 8000, 36, 2, 4, 3, 0, 0), (64, 8000, 36, 4, 4, 3, 0, 1), (128, 4000, 40, 1, 4, 4, 0, 0),
    (128, 8000, 40, 1, 4, 4, 0, 1), (128, 8000, 40, 1, 2, 2, 0, 0), (128, 8000, 48, 1, 4, 4, 0, 0),
    (128, 8000, 48, 4, 2, 2, 0, 1), (64, 8000, 48, 4, 2, 2, 0, 0), (64, 8000, 40, 4, 4, 4, 1, 1),
    (64, 8000, 36, 1, 3, 2, 0, 0), (64, 1000, 36, 1, 3, 2, 0, 1), (64, 8000, 40, 1, 3, 2, 0, 1),
    (64, 8000, 48, 1, 3, 2, 0, 0), (128, 8000, 8, 1, 4, 4, 1, 0), (128, 8200, 8, 1, 4, 4, 1, 1),
    (64, 16000, 12, 1, 4, 4, 1, 0), (64, 32000, 12, 1, 4, 4, 1, 1), (64, 32000, 12, 1, 2, 2, 1, 0),
    (64, 7000, 32, 1, 2, 2, 1, 0), (64, 8000, 32, 1, 2, 2, 1, 1), (128, 6000, 16, 1, 2, 2, 1, 0),
    (128, 8000, 16, 1, 2, 2, 1, 1), (64, 16000, 20, 1, 4, 4, 1, 1), (64, 16000, 20, 1, 2, 2, 1, 0),
    (128, 65536, 1, 1, 2, 2, 1, 1), (64, 140000, 1, 1, 4, 4, 1, 1),
]


@pytest.mark.parametrize("dim,tokens,kv,nq,kb,vb,head_major,codes", ROUTES)
def test_route(built_library, dim, tokens, kv, nq, kb, vb, head_major, codes):
    got = ctypes.c_uint32(7)
    assert _lib.load().pitch_selftest_attention_route(dim, tokens, kv, nq, kb, vb, head_major, 256, ctypes.byref(got)) == 0
    assert got.value == codes


@pytest.mark.parametrize("dim", [64, 128])
def test_one_workgroup_up_to_twelve_tiles(split, dim):
    """A KV head of up to 12 tiles of 64 tokens (key-bias: 4) is one workgroup; longer ones are split, since a fourth
    wave per SIMD, or a third round of eight waves, takes longer than the second launch."""
    for kv in (1, 8, 24):
        for bias, most in ((0, 768), (1, 256)):
            assert split(dim, most, kv, bias, 256)[1] == 1
            chunk, chunks, _, _ = split(dim, most + 1, kv, bias, 256)
            assert chunks > 1 and chunk <= 128


def test_workspace_is_what_the_size_query_says(split):
    lib = _lib.load()
    cfg = _lib.PitchConfigC(0, 128, 4, 1)
    size = ctypes.c_uint64()
    for kv in (1, 3, 64):
        for tokens in (1, 1000, 70000):
            desc = _lib.PitchAttentionDescC(1, kv, tokens, 1, tokens, 1.0, 0)
            assert lib.pitch_attention_workspace_size(ctypes.byref(cfg), ctypes.byref(cfg), ctypes.byref(desc),
                                                      ctypes.byref(size)) == 0
            assert size.value == 4 * split(128, tokens, kv, 0, 256)[3]
