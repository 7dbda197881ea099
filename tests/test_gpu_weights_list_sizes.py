"""Coarse weights over the lists of pools on both sides of the number of CUs (256): an image then has a block of 1024 or of
512 threads.  Broad posteriors: lists past 8192 entries, more candidates than their buffer (whether another pass can
collect them is read from the buckets) and lists whose candidates fit.  Against the full pose term's weights: the same
FP64 expressions over the same values, so integers are equal and sums differ by the order of at most 33408 additions
(2^-53 each): 1e-11."""
import numpy as np
import pytest

from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,snr", [(256, 0.02), (257, 0.02), (257, 0.2), (40, 1e-6)])
def test_list_blocks_match_the_full_pose_term(engine, n, snr):
    print(f"[weights list n={n} snr={snr}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=16, K=2, order=1, offset_range=3.0, n=n,
                                        snr=snr, seed=7, sigma_offset=4.0)
    synth.load_engine(engine, prob)
    out = {}
    try:
        for mode in ("full", "list"):
            engine.set_coarse_mode(mode)
            engine.reset_sums()
            r = engine.expectation(batch)
            out[mode] = (r, engine.get_sums())
        st = engine.coarse_stats()
        print("  list_max", st["list_max"], "nr_sign", int(r["nr_sign"].min()), int(r["nr_sign"].max()), flush=True)
        assert st["mode"] == 0 and st["list_max"] > 8192
    finally:
        engine.set_coarse_mode("list")
    (rf, sf), (r, s) = out["full"], out["list"]
    for k in ("argmax", "nr_sign", "min_diff2", "min_diff2_coarse"):
        np.testing.assert_array_equal(r[k], rf[k], err_msg=k)
    for k in ("sum_weight_coarse", "sum_weight", "sig_weight_coarse", "sig_weight"):
        np.testing.assert_allclose(r[k], rf[k], rtol=1e-11, err_msg=k)
    for k in ("wsum_pdf_class", "wsum_sigma2_noise", "wsum_scalars"):
        np.testing.assert_allclose(s[k], sf[k], rtol=1e-10, err_msg=k)
