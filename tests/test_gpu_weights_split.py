"""Coarse weights of broad posteriors: lists below and above the length from which they are scanned by several
blocks (8192), with partly filled last parts, more entries inside the window than the candidate list holds, and
more significant samples than the keys hold (the weights then run twice over the same lists).  The list form
must agree with the full pose term's (one block scanning every entry): the same FP64 expressions over the same
values, so integers are equal and sums differ by the order of at most 33408 additions (2^-53 each): 1e-11."""
import numpy as np
import pytest

from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,rng,precision,snr", [(1, 2.0, "fp32", 0.02), (1, 3.0, "fp32", 0.02), (2, 3.0, "fp32", 0.2),
                                                 (2, 3.0, "fp16", 0.02), (1, 3.0, "bf16", 0.002), (2, 3.0, "fp32", 1e-6)])
def test_long_lists_match_the_full_pose_term(engine, K, rng, precision, snr):
    print(f"[weights split K={K} range={rng} {precision} snr={snr}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=16, K=K, order=1, offset_range=rng, n=5,
                                        snr=snr, seed=7, sigma_offset=4.0)
    synth.load_engine(engine, prob, precision=precision)
    out = {}
    for mode in ("full", "list", "list"):  # the second list pass starts from the histograms the first one left
        engine.set_coarse_mode(mode)
        engine.reset_sums()
        r = engine.expectation(batch)
        out.setdefault(mode, []).append((r, engine.get_sums()))
        if mode == "list":
            st = engine.coarse_stats()
            print("  list_max", st["list_max"], "nr_sign max", int(r["nr_sign"].max()), flush=True)
    engine.set_coarse_mode("list")
    (rf, sf), = out["full"]
    for r, s in out["list"]:
        for k in ("argmax", "nr_sign", "min_diff2", "min_diff2_coarse"):
            np.testing.assert_array_equal(r[k], rf[k], err_msg=k)
        for k in ("sum_weight_coarse", "sum_weight", "sig_weight_coarse", "sig_weight"):
            np.testing.assert_allclose(r[k], rf[k], rtol=1e-11, err_msg=k)
        for k in ("wsum_pdf_class", "wsum_sigma2_noise", "wsum_scalars"):
            np.testing.assert_allclose(s[k], sf[k], rtol=1e-10, err_msg=k)
