"""Device-driven pools whose images have many times more significant samples than the key cap: nothing may be emitted for
such an image (the task and block buffers hold cap entries an image), the pool aborts on the device and its host-synchronised
rerun gives the host-synchronised results; later device-driven pools of the context still agree.  All images past the
cap, and one image alone among others that fit; FP32 and a mixed arm, whose marked samples are emitted too."""
import numpy as np
import pytest

from rome_amd import synth
from test_gpu_exec import _pool, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,cap,narrow", [("fp32", 16, False), ("fp16", 16, False), ("fp32", 300, True)])
def test_counts_far_past_the_cap(engine, prec, cap, narrow):
    prob, batch, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=16, K=2, order=1, n=4, snr=0.02, seed=5)
    if narrow:  # the last image stays broad
        sharp, sb, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=16, K=2, order=1, n=4, snr=2.0, seed=5)
        for k in ("fmask_re", "fmask_im"):
            batch[k][:3] = sb[k][:3] * np.sqrt(np.mean(sharp["sigma2_noise"]) ** -1 * np.mean(prob["sigma2_noise"]))
    print(f"[key overflow {prec} cap={cap} narrow={narrow}]", flush=True)
    try:
        host = _pool(engine, prob, batch, prec, "host")
        nr = host[0]["nr_sign"]
        print("  nr_sign", nr, flush=True)
        assert nr.max() > 1.1 * cap and (not narrow or nr.min() <= cap)
        engine.set_significance_cap(cap)
        r = _pool(engine, prob, batch, prec, "device")
        assert r[3]["last"] == 1 | 8, r[3]
        _same(r, host, "rerun")
        engine.set_significance_cap(8192)
        r = _pool(engine, prob, batch, prec, "device")
        assert r[3]["last"] == 1 or prec != "fp32", r[3]  # (a mixed arm marks more samples than are significant)
        _same(r, host, "device-driven after it")
    finally:
        engine.set_significance_cap(-1)
        engine.set_execution("graph")
