"""2D backprojection by bands where one class takes most of the images: the blocks of a band follow the classes' slices.

Against the FP64 oracle (several partial bands for one class, one or none for the others; two bands of 100^2 images;
device-driven and host-synchronised), a grid point being an FP32 sum of at most a few thousand products: 1e-5 relative
L2, as for equal classes.  And the stage takes about as long as with that class alone: with as many blocks for every
class it took 16 times as long (20 classes of 200 images)."""
import numpy as np
import pytest

import oracle as O
from rome_amd import synth

pytestmark = pytest.mark.gpu


def _one_class(prob, k, share=1.0):
    w = np.full(prob["nr_classes"], (1 - share) / max(prob["nr_classes"] - 1, 1) + 1e-30)
    w[k] = share
    prob["pdf_class"] = w / w.sum()
    prob["pdf_direction"] = prob["pdf_class"].reshape(-1, 1) * np.ones(np.shape(prob["pdf_direction"])) \
        / np.shape(prob["pdf_direction"])[1]


@pytest.mark.parametrize("ori,K,n,over,mode", [(64, 4, 6, 0, "host"), (64, 5, 12, 1, "device"), (100, 3, 5, 1, "host"),
                                               (64, 1, 2, 1, "device")])
def test_unequal_classes_match_the_oracle(engine, ori, K, n, over, mode):
    print(f"[bp classes ori={ori} K={K} n={n} over={over} {mode}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=False, ori=ori, current=ori, coarse=ori if not over else 24, K=K,
                                        psi_step=10.0, offset_range=2.0, oversampling=over, n=n, snr=0.004, seed=K + n)
    _one_class(prob, K - 1, 0.9 if K > 3 else 1.0)
    ref = O.estep(prob, batch)
    try:
        synth.load_engine(engine, prob)
        engine.set_execution(mode)
        engine.reset_sums()
        engine.expectation(batch)
        print("  tasks", engine.batch_stats()["tasks"], engine.execution_stats()["last"], flush=True)
    finally:
        engine.set_execution("graph")
    for k in range(K):
        dg, wg = engine.get_backprojector(k)
        od, ow = np.asarray(ref["bp_data"][k]), np.asarray(ref["bp_weight"][k])
        assert np.linalg.norm(dg - od) <= 1e-5 * np.linalg.norm(od), k
        assert np.linalg.norm(wg - ow) <= 1e-5 * np.linalg.norm(ow), k


def test_time_follows_the_slices(engine):
    ms = {}
    for K in (1, 20):
        prob, batch, _ = synth.make_problem(is3d=False, ori=64, current=64, coarse=24, K=K, psi_step=10.0,
                                            offset_range=3.0, oversampling=1, n=200, snr=0.004, seed=1)
        _one_class(prob, 0)
        synth.load_engine(engine, prob)
        engine.set_execution("host")
        try:
            engine.expectation(batch)
            t = []
            for _ in range(5):
                engine.set_profiling(True)
                engine.reset_sums()
                engine.expectation(batch)
                t.append(engine.profile()["backproject"][0])
            ms[K] = (float(np.median(t)), engine.batch_stats()["tasks"])
        finally:
            engine.set_profiling(False)
            engine.set_execution("graph")
    print("[bp classes] ms, tasks by classes", ms, flush=True)
    per = {K: v[0] / v[1] for K, v in ms.items()}
    assert per[20] <= 4 * per[1]
