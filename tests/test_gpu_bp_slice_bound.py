"""The slice buffer of 2D pools is bounded: pools of more slices take the direct scatter, on the device's own decision
(device-driven) or the host's, and either side of the switch adds a pool exactly once.

Images of 200^2 with posteriors over nearly every rotation: device-driven the buffer holds 4.2 thousand slices (512 MB),
which 10 such images stay below and 24 exceed; host-synchronised 34 thousand (4 GB), which 150 images exceed.  Grids are FP32
sums of one value a slice in different orders: 1e-5 relative L2; FP64 sums 1e-10."""
import numpy as np
import pytest

from rome_amd import synth

pytestmark = pytest.mark.gpu


def _problem(n):
    return synth.make_problem(is3d=False, ori=200, current=200, coarse=16, K=2, psi_step=5.0, offset_range=2.0,
                              oversampling=1, n=n, snr=2e-5, seed=21)[:2]


def _run(engine, batch, mode, parts=1):
    engine.set_execution(mode)
    engine.reset_sums()
    n, slices, last = batch["n"], 0, []
    for p in range(parts):
        a, b = n * p // parts, n * (p + 1) // parts
        engine.expectation({k: v[a:b] if isinstance(v, np.ndarray) and len(v) == n else (b - a if k == "n" else v)
                            for k, v in batch.items()})
        slices = max(slices, 2 * engine.batch_stats()["tasks"])
        last.append(engine.execution_stats()["last"])
    return [engine.get_backprojector(k) for k in range(2)], engine.get_sums(), slices, last


def _same(a, b, what):
    for (da, wa), (db, wb) in zip(a[0], b[0]):
        assert np.linalg.norm(da - db) <= 1e-5 * np.linalg.norm(db), what
        assert np.linalg.norm(wa - wb) <= 1e-5 * np.linalg.norm(wb), what
    for k in a[1]:
        np.testing.assert_allclose(a[1][k], b[1][k], rtol=1e-10, atol=1e-300, err_msg=f"{what}: {k}")


@pytest.mark.parametrize("n", [10, 24])
def test_device_driven_switch(engine, n):
    prob, batch = _problem(n)
    synth.load_engine(engine, prob)
    try:
        engine.set_significance_cap(8192)
        host = _run(engine, batch, "host")
        print(f"[slice bound] n={n} slices={host[2]}", flush=True)
        cap = max((512 << 20) // (8 * engine.batch_stats()["Pf"]), n * 64)
        assert host[2] < cap if n == 10 else host[2] > cap, (host[2], cap)
        for rep in range(2):
            dev = _run(engine, batch, "device")
            assert dev[3] == [1], dev[3]
            _same(dev, host, f"device-driven {rep}")
    finally:
        engine.set_significance_cap(-1)
        engine.set_execution("graph")


def test_host_bound(engine):
    import torch
    prob, batch = _problem(150)
    synth.load_engine(engine, prob)
    try:
        engine.set_significance_cap(8192)
        few = _run(engine, batch, "host", parts=10)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        whole = _run(engine, batch, "host")
        torch.cuda.synchronize()
        used = free - torch.cuda.mem_get_info()[0]
        Pf = engine.batch_stats()["Pf"]
        print(f"[slice bound] slices {few[2]} {whole[2]}, {8e-9 * whole[2] * Pf:.2f} GB, grown by {used / 1e9:.2f} GB", flush=True)
        assert whole[2] > (4 << 30) // (8 * Pf) > few[2]
        _same(whole, few, "past the bound")
        assert used < 2 << 30
    finally:
        engine.set_significance_cap(-1)
        engine.set_execution("graph")
