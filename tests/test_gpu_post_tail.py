"""Post slices past the first launch of a device-driven pool: without the totals of earlier pools the launch covers four
tasks an image and the tail nearly all of the rest.  Its sums are those of the host-synchronised pool to the order of the
atomic additions, with the default grid and with eight blocks, and the stage stays within 2.2 times the time it takes when
the first launch covers the pool (a work counter per range made it 4 times; 1.1 strided).  300 given coarse samples of
every image, most of whose fine slices have no significant sample."""
import numpy as np
import pytest

from rome_amd import synth
from test_gpu_exec import _same
from test_gpu_fine_given import _device_batch, _run_given

pytestmark = pytest.mark.gpu


def test_tail(engine):
    import torch
    prob, batch, _ = synth.make_problem(is3d=True, ori=128, current=128, coarse=16, K=1, order=1, offset_range=2.0,
                                        n=64, snr=0.05, seed=11)
    n, cap = batch["n"], 300
    MT = prob["nr_dir"] * prob["nr_psi"] * prob["nr_trans"]
    rng = np.random.default_rng(12)
    keys = torch.tensor(np.stack([rng.permutation(MT)[:cap] for _ in range(n)]).astype(np.int32), device="cuda")
    cnt = torch.full((n,), cap, dtype=torch.int32, device="cuda")
    t = _device_batch(batch)
    torch.cuda.synchronize()
    synth.load_engine(engine, prob)

    def pool(mode):
        engine.set_execution(mode)
        engine.reset_sums()
        r = _run_given(engine, t, n, keys, cnt, cap)
        for k in ("min_diff2_coarse", "sum_weight_coarse", "sig_weight_coarse"):
            r[k] = np.zeros(n)  # NaN
        return r, engine.get_sums(), [engine.get_backprojector(0)], engine.execution_stats()

    try:
        host = pool("host")
        tasks = engine.batch_stats()["tasks"]
        print("[post tail] tasks", tasks, flush=True)
        assert tasks > 16 * n
        for grid in (0, 8):
            engine.set_persistent_grids([0, 0, grid, 0])
            dev = pool("device")
            assert dev[3]["last"] == 1, dev[3]
            _same(dev, host, f"tail of {grid} blocks")
        ms = {}
        for known in (False, True):
            v = []
            for _ in range(6):
                if not known:
                    engine.set_persistent_grids([0, 0, 0, 0])
                engine.set_profiling(True)
                pool("device")
                v.append(engine.profile()["post"][0])
            ms[known] = float(np.median(v[1:]))
        print("[post tail] ms without and with known totals", ms, flush=True)
        assert ms[False] <= 2.2 * ms[True]
    finally:
        engine.set_profiling(False)
        engine.set_persistent_grids([0, 0, 0, 0])
        engine.set_execution("graph")
