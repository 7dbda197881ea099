"""2D backprojection by bands of grid rows held in LDS, against the FP64 oracle's E-step: one band and one part (sums
added to the grids directly), several parts a class (partial sums), grids of more rows than LDS holds (two bands),
one and both passes.  Two pools of the same images double the sums, the second one device-driven where the engine
does that.  A grid point sums FP32 products, at most a few thousand: 1e-5 relative L2, as for the 3D grids."""
import numpy as np
import pytest

import oracle as O
from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ori,cur,K,n,over", [(32, 24, 2, 3, 1), (64, 64, 3, 40, 0), (64, 50, 2, 17, 1),
                                              (100, 100, 1, 24, 1), (100, 92, 2, 5, 0)])
def test_bands_match_the_oracle(engine, ori, cur, K, n, over):
    print(f"[bp bands ori={ori} cur={cur} K={K} n={n} over={over}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=False, ori=ori, current=cur, coarse=cur if not over else min(cur, 24), K=K,
                                        psi_step=30.0, offset_range=1.0, oversampling=over, n=n, snr=0.3, seed=ori + n)
    ref = O.estep(prob, batch)
    synth.load_engine(engine, prob)
    engine.reset_sums()
    for _ in range(2):
        engine.expectation(batch)
    for k in range(K):
        dg, wg = engine.get_backprojector(k)
        od, ow = 2 * np.asarray(ref["bp_data"][k]), 2 * np.asarray(ref["bp_weight"][k])
        assert np.linalg.norm(dg - od) <= 1e-5 * np.linalg.norm(od), k
        assert np.linalg.norm(wg - ow) <= 1e-5 * np.linalg.norm(ow), k
