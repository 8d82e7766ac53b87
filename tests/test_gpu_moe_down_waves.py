"""The MoE down projection of few tokens with 4, 6 and 8 wavefronts per block,
against the CPU oracle.
"""
import numpy as np
import pytest

from conftest import PROMPT_SEED
from strasgpt_amd import synth

pytestmark = pytest.mark.gpu


# width, expert width, top-k, {tokens per call: wavefronts}: widths that are no
# multiple of a block's 16 rows, one and two tokens with 8, two with 6, and
# top-8 rows of 2880 (more slots and blocks than one unrolled pass holds)
@pytest.mark.parametrize("dim,hidden,topk,waves", [(3104, 96, 4, {1: 8, 2: 4}), (2016, 96, 2, {1: 4, 2: 8, 3: 4}),
                                                   (1504, 96, 3, {1: 4, 2: 6, 5: 4}), (4064, 2880, 8, {1: 8})])
def test_down_waves(dim, hidden, topk, waves, tmp_path):
    """Prompts of so many tokens, and a token decoded after each: logits at the
    parity bar (1e-3 + 2e-2 |value|), the launch rule's wavefronts as stated."""
    from oracle import oracle as orc
    from strasgpt_amd import runtime as rt
    shp = synth.ModelShape("down", dim, hidden, 1, 4, 2, 32, 256, 150000.0, 1e-5, 8, 8, untied=True, experts=8,
                           experts_per_tok=topk, model_type="stras_moe", std=0.02)
    d = str(tmp_path / "down")
    synth.write_model(shp, d, seed=13)
    oracle = orc.OracleModel(d, threads=16)
    with rt.Transformer(d) as t:
        for tokens, want in waves.items():
            assert t._lib.strasgpt_kbench_moe_down_waves(dim, tokens) == want
            prompt = synth.prompt_tokens(shp.vocab, tokens + 1, PROMPT_SEED + tokens)
            oracle.reset()
            t.reset()
            for piece in (prompt[:tokens], prompt[tokens:]):
                ref, got = oracle.predict(piece, len(piece)), t.predict(piece, len(piece))
                err = float(np.abs(got - ref).max())
                print(f"[down waves] N={dim} top-{topk}, {len(piece)} tokens: max |error| {err:.3g} of "
                      f"{np.abs(ref).max():.3g}", flush=True)
                np.testing.assert_allclose(got, ref, rtol=2e-2, atol=1e-3)
