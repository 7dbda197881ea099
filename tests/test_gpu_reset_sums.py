"""rome_reset_sums clears every sum with one kernel (blocks of 4096 words, whole and partial ones, arrays of a few
words): after it nothing is left of a pool, and the pool's sums come out as in a fresh start."""
import numpy as np
import pytest

from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("is3d,ori,K,groups", [(False, 16, 1, 1), (False, 44, 7, 3), (True, 20, 3, 2), (True, 32, 2, 5)])
def test_reset_clears_all_sums(engine, is3d, ori, K, groups):
    prob, batch, _ = synth.make_problem(is3d=is3d, ori=ori, current=ori, coarse=min(ori, 16), K=K, psi_step=30.0,
                                        offset_range=1.0, n=6, nr_groups=groups, snr=0.3, seed=ori + K)
    synth.load_engine(engine, prob)

    def state():
        return [*engine.get_sums().values(), *(a for k in range(K) for a in engine.get_backprojector(k))]

    engine.reset_sums()
    assert not any(np.any(a) for a in state())
    engine.expectation(batch)
    first = state()
    engine.expectation(batch)
    engine.reset_sums()
    assert not any(np.any(a) for a in state())
    engine.expectation(batch)
    for a, b in zip(first, state()):  # FP32 / FP64 atomics: sums of a few thousand terms in another order
        np.testing.assert_allclose(b, a, rtol=1e-4, atol=1e-5 * np.max(np.abs(a), initial=0.0))
