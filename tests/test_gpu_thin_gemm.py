"""Prefill GEMMs of short prompts (at most 128 rows): one row tile of 16, 32,
48, 64, 96 or 128 rows over 64 or 128 columns, against the CPU oracle.
"""
import numpy as np
import pytest

from conftest import PROMPT_SEED
from strasgpt_amd import synth

pytestmark = pytest.mark.gpu

# Wide outputs (SwiGLU and QKV on 128-wide tiles at every row tile; the O and
# down projections on 64-wide ones with up to 16 splits), and narrow ones
# (every projection on 64-wide tiles, the O and down with 8 splits).
SHAPES = [
    synth.ModelShape("thin-wide", 512, 16384, 1, 64, 8, 128, 352, 10000.0, 1e-5, 8, 8, ctx=160, std=0.05),
    synth.ModelShape("thin-narrow", 2048, 2048, 1, 16, 4, 64, 352, 10000.0, 1e-6, 8, 8, qk_norm=True, ctx=160,
                     std=0.03),
]


@pytest.mark.parametrize("shp", SHAPES, ids=lambda s: s.name)
def test_thin_gemm_rows(shp, tmp_path):
    """Lengths around every row tile's edge, each row's logits compared, at
    the parity bar (1e-3 + 2e-2 |value|)."""
    from oracle import oracle as orc
    from strasgpt_amd import runtime as rt
    d = str(tmp_path / shp.name)
    synth.write_model(shp, d, seed=11)
    om = orc.OracleModel(d, threads=16)
    prompt = synth.prompt_tokens(shp.vocab, 129, PROMPT_SEED)
    want = om.predict(prompt, len(prompt))
    with rt.Transformer(d) as t:
        for T in (9, 16, 17, 32, 33, 47, 48, 49, 64, 65, 95, 96, 97, 128, 129):
            t.reset()
            got = t.predict(prompt[:T], T)
            err = float(np.abs(got - want[:T]).max())
            print(f"[thin gemm] {shp.name} {T} rows: max |error| {err:.3g} of {np.abs(want[:T]).max():.3g}", flush=True)
            np.testing.assert_allclose(got, want[:T], rtol=2e-2, atol=1e-3)


@pytest.mark.parametrize("kv", ["fp32", "bf16"])
def test_short_prompts_continued(kv, tmp_path):
    """A prompt given in ragged pieces (each sums its split QKV products, and
    writes its cache and plane rows, from a position that is no multiple of
    32) ends in the logits of the same prompt in one call: within 2e-3 of
    their largest magnitude (sums in another order; with the bf16 cache a key
    or value near a rounding edge goes to the other neighbour)."""
    from strasgpt_amd import runtime as rt
    shp = SHAPES[1]
    d = str(tmp_path / shp.name)
    synth.write_model(shp, d, seed=11)
    prompt = synth.prompt_tokens(shp.vocab, 121, PROMPT_SEED)
    with rt.Transformer(d) as t:
        if kv == "bf16":
            t.set_kv_cache_format(rt.KV_BF16)
        want = t.predict(prompt)[0]
        t.reset()
        at = 0
        for n in (5, 21, 1, 45, 33, 16):
            got = t.predict(prompt[at:at + n])[0]
            at += n
    assert at == len(prompt)
    err = float(np.abs(got - want).max())
    print(f"[thin gemm] continued, {kv} cache: {err:.3g} of {np.abs(want).max():.3g}", flush=True)
    assert err < 2e-3 * float(np.abs(want).max())


@pytest.mark.parametrize("kv", ["fp32", "bf16"])
def test_short_prompts_after_long_context(kv, tmp_path):
    """Few queries after a context of 16 key tiles and more: the prefill
    attention split over key ranges (empty last ranges: 65 tiles in 16 ranges
    of 5; a range that some queries of a block see nothing of; 2 to 8 rows with
    fp32 outputs), against the same prompt in one call, whose query blocks fill
    the GPU and are not split (both as the launch rule says). Bound as above."""
    from strasgpt_amd import runtime as rt
    shp = synth.dataclasses.replace(SHAPES[1], name="thin-context", heads=32, kv_heads=8, ctx=2100)
    d = str(tmp_path / shp.name)
    synth.write_model(shp, d, seed=11)
    prompt = synth.prompt_tokens(shp.vocab, 2059, PROMPT_SEED)

    def ranges(queries, keys):
        return rt.lib().strasgpt_kbench_attention_ranges(shp.heads, shp.head_dim, queries, keys)

    with rt.Transformer(d) as t:
        if kv == "bf16":
            t.set_kv_cache_format(rt.KV_BF16)
        for cuts, split in (((600, 120, 45, 3, 9), (1, 5, 6, 6, 6)), ((511, 2), (1, 4)),
                            ((700, 90, 64), (1, 6, 6)), ((2050, 9), (1, 16))):
            assert ranges(sum(cuts), sum(cuts)) == 1
            t.reset()
            want = t.predict(prompt[:sum(cuts)])[0]
            t.reset()
            at = 0
            for n, r in zip(cuts, split):
                assert ranges(n, at + n) == r
                got = t.predict(prompt[at:at + n])[0]
                at += n
            err = float(np.abs(got - want).max())
            print(f"[thin gemm] {cuts}, {kv} cache: {err:.3g} of {np.abs(want).max():.3g}", flush=True)
            assert err < 2e-3 * float(np.abs(want).max())
