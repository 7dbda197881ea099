"""Coarse operands written in groups of 8 images x 32 pixels: pools of 1, 7, 8, 9 and 130 images (group edges, the
padding after the last image past a second 128-image block) and 13 / 29 translations.  Every entry of the coarse
pose term is compared with the FP64 oracle: FP32 operands and accumulation over at most 2 x 312 products, 1e-5
relative as in the parity tests."""
import numpy as np
import pytest

import oracle as O
from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rng,coarse", [(1, 2.0, 16), (7, 3.0, 18), (8, 2.0, 16), (9, 3.0, 22), (130, 2.0, 16)])
def test_coarse_operands(engine, n, rng, coarse):
    print(f"[prep coarse n={n} range={rng} coarse={coarse}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=coarse, K=1, order=0, offset_range=rng,
                                        n=n, snr=0.5, seed=n)
    synth.load_engine(engine, prob)
    engine.set_coarse_mode("full")
    r = engine.expectation(batch)
    got = engine.get_coarse_diff2(n)
    engine.set_coarse_mode("list")
    ref = O.estep(prob, batch, dump_coarse=True)
    want = ref["coarse_diff2"].reshape(got.shape)
    assert np.max(np.abs(got - want) / want) < 1e-5
    np.testing.assert_allclose(r["min_diff2_coarse"], ref["min_diff2_coarse"], rtol=1e-5)
