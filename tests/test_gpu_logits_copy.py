"""Large logits on their way to the caller: above 4 MiB through the two halves
of a pinned staging buffer, by several threads, or directly where the caller's
buffer is pinned itself.
"""
import ctypes

import numpy as np
import pytest

from conftest import PROMPT_SEED
from strasgpt_amd import synth

pytestmark = pytest.mark.gpu


# rows x vocabulary: just 4 MiB (no staging), a little more (a second half of
# 128 KiB), two whole halves, three pieces with the first half reused (the last
# piece by several threads), and four with both reused (the last of 13 KiB)
@pytest.mark.parametrize("vocab,rows", [(32768, 32), (32768, 33), (32768, 64), (32003, 82), (31491, 100)])
def test_large_logits_reach_the_caller(vocab, rows, tmp_path):
    """Every row against the CPU oracle (at the parity bar, 1e-3 + 2e-2
    |value|: a misplaced or stale piece is off by the values themselves), in
    fresh, unaligned and pinned buffers bit for bit the same, nothing beside
    them written; a second prompt through the same halves likewise."""
    from oracle import oracle as orc
    from strasgpt_amd import runtime as rt
    shp = synth.ModelShape("copy", 64, 96, 1, 4, 1, 32, vocab, 500000.0, 1e-5, 100, 4, ctx=104, std=0.25)
    d = str(tmp_path / "copy")
    synth.write_model(shp, d, seed=11)
    oracle = orc.OracleModel(d, threads=16)
    n = rows * vocab
    hip = rt.lib()  # (its HIP runtime's functions are found through it)
    address = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(address), ctypes.c_size_t(4 * (n + 6)), 0) == 0
    pinned = np.ctypeslib.as_array(ctypes.cast(address, ctypes.POINTER(ctypes.c_float)), (n + 6,))
    with rt.Transformer(d) as t:
        def into(buffer, at, prompt):
            t.reset()
            t._lib.transformer_predict(t._t, len(prompt), rt._ints(prompt), rows,
                                       ctypes.cast(buffer + 4 * at, ctypes.POINTER(ctypes.c_float)))

        for seed in (PROMPT_SEED, PROMPT_SEED + 1):
            prompt = synth.prompt_tokens(vocab, 100, seed)
            oracle.reset()
            want = oracle.predict(prompt, rows)
            fresh = np.full(n + 6, -7.0, np.float32)
            into(fresh.ctypes.data, 3, prompt)  # unaligned by 12 bytes
            got = fresh[3:3 + n]
            err = float(np.abs(got.reshape(rows, vocab) - want).max())
            print(f"[logits copy] {rows} x {vocab}: max |error| {err:.3g}", flush=True)
            np.testing.assert_allclose(got.reshape(rows, vocab), want, rtol=2e-2, atol=1e-3)
            assert (fresh[:3] == -7.0).all() and (fresh[3 + n:] == -7.0).all()
            pinned[:] = -7.0
            into(address.value, 3, prompt)
            np.testing.assert_array_equal(pinned[3:3 + n], got)
            assert (pinned[:3] == -7.0).all() and (pinned[3 + n:] == -7.0).all()
            t.reset()
            np.testing.assert_array_equal(t.predict(prompt, rows).reshape(-1), got)
    assert hip.hipHostFree(address) == 0
