"""Fine weights of images on both sides of the split between blocks of 256 and of 1024 threads: 127, 128 and 129 given coarse
samples (4064, 4096 and 4128 fine ones), one and 700 in one pool, against the FP64 oracle with the same significance;
bars as for the other pools of given significance."""
import numpy as np
import pytest

import oracle as O
from rome_amd import synth
from test_gpu_fine_given import _device_batch, _run_given
from test_gpu_parity import _case, _check_lists, _check_sums

pytestmark = pytest.mark.gpu


def test_fine_weight_blocks(engine):
    import torch
    name, ne = "3d", 32
    prob, batch, truth = _case(name)
    n = batch["n"]
    MT = prob["nr_classes"] * prob["nr_dir"] * prob["nr_psi"] * prob["nr_trans"]
    want = [4096 // ne - 1, 4096 // ne, 4096 // ne + 1, 1, 700]
    counts = np.array([min(want[i % len(want)], MT) for i in range(n)], np.int32)
    keys, counts = synth.clustered_significance(prob, np.asarray(truth, float), counts)
    print(f"[fine weights {name}] counts={counts.tolist()} of {MT}", flush=True)
    assert np.any(counts * ne == 4096) and np.any(counts * ne > 4096)
    ref = O.estep(prob, dict(batch, coarse_sig_in=synth.significance_mask(prob, keys, counts)), dump_fine=True,
                  dump_fine_weight=True)
    t = _device_batch(batch)
    kt, ct = torch.tensor(keys, device="cuda"), torch.tensor(counts, device="cuda")
    torch.cuda.synchronize()
    try:
        for mode in ("host", "device"):
            synth.load_engine(engine, prob)
            engine.set_execution(mode)
            r = _run_given(engine, t, n, kt, ct, keys.shape[1])
            s = engine.get_sums()
            assert np.array_equal(r["nr_sign"], counts), mode
            _check_lists(engine, r, ref, n, f"{name} {mode}")
            _check_sums(r, s, ref, prob, engine, f"{name} {mode}")
    finally:
        engine.set_execution("graph")
