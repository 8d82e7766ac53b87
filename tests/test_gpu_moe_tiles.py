"""The grouped MXFP4 prefill GEMM's tilings: 16 or 32 slots in K steps of 128,
32 or 64 slots in K steps of 64.
"""
import numpy as np
import pytest

from conftest import PROMPT_SEED
from strasgpt_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,lengths", [("tiny-moe-long", (8, 9, 33, 64)), ("mid-moe", (8, 9, 21, 40))])
def test_moe_slot_tiles_bit_identical(name, lengths, tmp_path, monkeypatch):
    """Few slots per expert: tiles with 1 to 16 slots (row groups of 4 skipped
    by the activation DMA), rows of K = 2880 whose last step holds two of four
    blocks (mid-moe). The tiling changes no product and no order of a sum."""
    from strasgpt_amd import runtime as rt
    shp = synth.dataclasses.replace(synth.shape(name), ctx=max(lengths))
    d = str(tmp_path / name)
    synth.write_model(shp, d, seed=7)
    prompt = synth.prompt_tokens(shp.vocab, max(lengths), PROMPT_SEED)
    with rt.Transformer(d) as t:
        for T in lengths:
            got = {}
            for tile in ("16", "32", "64"):
                monkeypatch.setenv("STRASGPT_MOE_TILE", tile)
                t.reset()
                got[tile] = t.predict(prompt[:T], T)
            np.testing.assert_array_equal(got["16"], got["64"])
            np.testing.assert_array_equal(got["32"], got["64"])


def test_moe_slot_tiles_wide_code_rows(tmp_path, monkeypatch):
    """Code rows 512 and 1024 bytes apart (inputs of 1024 and 2048), for which
    32 slots run in K steps of 64: bit-identical to 16 and 64 slots, and at the
    parity bar (1e-3 + 2e-2 |value|) from the oracle. Tiles with 1 to 32 slots."""
    from oracle import oracle as orc
    from strasgpt_amd import runtime as rt
    shp = synth.ModelShape("wide-codes", 1024, 2048, 1, 4, 2, 32, 256, 150000.0, 1e-5, 8, 8, untied=True, experts=8,
                           experts_per_tok=2, model_type="stras_moe", std=0.02, ctx=130)
    d = str(tmp_path / "wide-codes")
    synth.write_model(shp, d, seed=7)
    prompt = synth.prompt_tokens(shp.vocab, 130, PROMPT_SEED)
    want = orc.OracleModel(d, threads=16).predict(prompt, len(prompt))
    with rt.Transformer(d) as t:
        for T in (9, 40, 130):
            got = {}
            for tile in ("16", "32", "64"):
                monkeypatch.setenv("STRASGPT_MOE_TILE", tile)
                t.reset()
                got[tile] = t.predict(prompt[:T], T)
                np.testing.assert_allclose(got[tile], want[:T], rtol=2e-2, atol=1e-3)
            np.testing.assert_array_equal(got["16"], got["64"])
            np.testing.assert_array_equal(got["32"], got["64"])
