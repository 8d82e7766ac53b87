"""The prefill's launch rules over their whole ranges (host arithmetic: no GPU)."""
import ctypes
import os

import pytest

from strasgpt_amd import _paths, synth

pytestmark = pytest.mark.skipif(not os.path.exists(_paths.hip_lib()), reason="library not built")


BF16X2, BF16 = 0, 1


def gemm_splits(M, N, K, precision=BF16X2):
    """(splits as the QKV projection, as the O or down projection)."""
    from strasgpt_amd import runtime as rt
    qkv, other = ctypes.c_int(), ctypes.c_int()
    assert rt.lib().strasgpt_kbench_gemm_splits(M, N, K, precision, ctypes.byref(qkv), ctypes.byref(other)) == 0
    return qkv.value, other.value


def projections(shp):
    """(N, K) of the QKV, O and down projections."""
    hd = shp.head_dim
    return ((shp.heads + 2 * shp.kv_heads) * hd, shp.dim), (shp.dim, shp.heads * hd), (shp.dim, shp.hidden)


@pytest.mark.parametrize("name", sorted(synth.PRESETS))
def test_thin_row_splits_fill_the_cus(name):
    """Prompts of 9 to 64 rows, every benchmark shape: the thin tiles are at
    most 128 columns wide, so a QKV projection of fewer than 128 of them leaves
    half of the 256 CUs without a block unless it is split; no length is
    excepted, and a projection takes the same count wherever the split sums
    serve both."""
    qkv, o, _ = projections(synth.shape(name))
    for M in range(9, 65):
        n, _ = gemm_splits(M, *qkv)
        assert n > 1 and (qkv[0] + 63) // 64 * n >= 128, (M, qkv, n)
        as_qkv, as_o = gemm_splits(M, *o)
        assert as_qkv == as_o, (M, o)


@pytest.mark.parametrize("name,qkv,o,down", [("llama3.2-1b", 8, 8, 8), ("qwen3-4b", 6, 8, 8), ("llama3.1-8b", 6, 8, 8),
                                             ("mistral-small-24b", 6, 7, 8), ("moe-mxfp4", 7, 8, None)])
def test_single_bf16_few_rows_square_counts(name, qkv, o, down):
    """Single bf16 operands at up to 32 rows run the square tiles and take
    the counts made for them, not the thin tiles' (fewer) ones."""
    shapes = projections(synth.shape(name))
    for M in (9, 16, 31, 32):
        assert gemm_splits(M, *shapes[0], BF16)[0] == qkv
        assert gemm_splits(M, *shapes[1], BF16)[1] == o
        if down:
            assert gemm_splits(M, *shapes[2], BF16)[1] == down


@pytest.mark.parametrize("precision", [BF16X2, BF16])
@pytest.mark.parametrize("name", sorted(synth.PRESETS))
def test_forced_tile_square_counts(name, precision, monkeypatch):
    """With a tile shape forced the square tiles run at any length: a split
    QKV projection of 33 to 128 rows has one round of 64 x 128 tiles (two per
    CU, at least three quarters of the 512 slots)."""
    monkeypatch.setenv("STRASGPT_GEMM_TILE", "64x128x64")
    qkv = projections(synth.shape(name))[0]
    for M in (33, 45, 64, 65, 96, 128):
        n, _ = gemm_splits(M, *qkv, precision)
        tiles = (qkv[0] + 127) // 128 * ((M + 63) // 64)
        assert n == 1 or 384 <= tiles * n <= 512, (M, n, tiles)


FEW, MANY = (16, 128), (64, 64)
MID, MID64 = (32, 128), (32, 64)


@pytest.mark.parametrize("N,K,pair,changes", [
    (2880, 2880, 1, [(1, FEW), (12, MID), (29, FEW), (37, MANY)]),  # code rows over all 16 L2 channels, wide
    (1280, 2560, 1, [(1, FEW), (37, MANY)]), (4096, 1536, 0, [(1, FEW), (37, MANY)]),
    (6000, 4800, 1, [(1, FEW), (12, MID), (29, FEW), (37, MID64)]),  # one block of 64 slots per CU
    (1024, 3072, 1, [(1, FEW), (23, MID64), (64, MANY)]), (1536, 5120, 1, [(1, FEW), (14, MID64)]),  # 8 channels
    (2048, 1024, 0, [(1, FEW), (37, MID64), (64, MANY)]),
    (768, 2048, 1, [(1, FEW), (17, MID64), (64, MANY)]), (1024, 6144, 1, [(1, FEW), (5, MID64)]),  # 4
    (1536, 4096, 1, [(1, FEW), (4, MID64), (24, MANY)])])  # 2
def test_moe_slot_tile(N, K, pair, changes, monkeypatch):
    """The grouped GEMM's tile at both sides of every change of the rule, with
    few and many experts; the environment variable forces the slots."""
    from strasgpt_amd import runtime as rt
    step = ctypes.c_int()

    def tile(slots, experts):
        return rt.lib().strasgpt_kbench_moe_slot_tile(slots, experts, N, K, pair, ctypes.byref(step)), step.value

    for experts in (8, 128):
        for (at, want), (end, _) in zip(changes, changes[1:] + [(400, None)]):
            assert tile(at * experts, experts) == want, (at, experts)
            assert tile(end * experts - 1, experts) == want, (end, experts)
    for forced in (16, 32, 64):
        monkeypatch.setenv("STRASGPT_MOE_TILE", str(forced))
        assert tile(8, 8)[0] == forced


@pytest.mark.parametrize("heads,hd,queries,keys,ranges", [
    (32, 128, 45, 4045, 16), (32, 128, 448, 4448, 2), (32, 128, 449, 4449, 1),  # blocks fill the slots
    (32, 128, 45, 480, 1), (32, 128, 45, 481, 4),  # 15 and 16 tiles
    (16, 64, 512, 512, 1), (24, 64, 512, 512, 1), (16, 64, 608, 608, 1), (16, 64, 640, 640, 3),  # 16, 19, 20 tiles
    (8, 64, 512, 512, 4), (11, 64, 512, 512, 4), (12, 64, 512, 512, 1), (14, 64, 520, 520, 1),  # 88, 96 and 126 pairs
    (16, 128, 512, 512, 4),  # longer steps
    (64, 128, 8192, 8192, 1), (1, 16, 1, 1, 1)])
def test_prefill_attention_ranges(heads, hd, queries, keys, ranges):
    """Both sides of each line of the rule. Short walks of 96 pairs and more
    with heads of 64 stay whole: their ranges were the slower form."""
    from strasgpt_amd import runtime as rt
    assert rt.lib().strasgpt_kbench_attention_ranges(heads, hd, queries, keys) == ranges
