"""The prefill's launch rules over their whole ranges (host arithmetic: no GPU)."""
import ctypes
import os

import pytest

from strasgpt_amd import _paths, synth

pytestmark = pytest.mark.skipif(not os.path.exists(_paths.hip_lib()), reason="library not built")


def gemm_splits(M, N, K):
    """(splits as the QKV projection, as the O or down projection)."""
    from strasgpt_amd import runtime as rt
    qkv, other = ctypes.c_int(), ctypes.c_int()
    assert rt.lib().strasgpt_kbench_gemm_splits(M, N, K, ctypes.byref(qkv), ctypes.byref(other)) == 0
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
