"""FP32 coarse terms at tile edges: rotation counts below, at and past 32 / 128 rows (the last tiles partly padding),
image counts past one 32-column block, and odd numbers of 16-k chunks, against the FP64 oracle's coarse minimum:
1e-5 relative, as for the E-step's minima elsewhere."""
import numpy as np
import pytest

import oracle as O
from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("psi,K,n,ori,over", [(45.0, 1, 1, 16, 0), (22.5, 2, 33, 24, 0), (10.0, 4, 5, 20, 1),
                                              (8.0, 3, 34, 32, 0), (5.0, 4, 3, 36, 1)])
def test_coarse_minimum(engine, psi, K, n, ori, over):
    print(f"[coarse edges psi={psi} K={K} n={n} ori={ori} over={over}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=False, ori=ori, current=ori, coarse=ori if not over else min(ori, 18), K=K,
                                        psi_step=psi, offset_range=1.0, oversampling=over, n=n, snr=0.3, seed=n + K)
    ref = O.estep(prob, batch)
    synth.load_engine(engine, prob)
    for mode in ("full", "list"):
        engine.set_coarse_mode(mode)
        engine.reset_sums()
        r = engine.expectation(batch)
        np.testing.assert_allclose(r["min_diff2"], ref["min_diff2"], rtol=1e-5, err_msg=mode)
        np.testing.assert_allclose(r["min_diff2_coarse"], ref["min_diff2_coarse"], rtol=1e-5, err_msg=mode)
    engine.set_coarse_mode("list")
