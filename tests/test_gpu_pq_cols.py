"""The paired cross term with resident columns takes pools of many columns; the full pose term always takes the tiled
kernel.  Both multiply in the same order, so their E values are the same and the results are held to what summing them
in another order can change: integers equal, sums of at most a few thousand terms to 1e-11.  96 and 64 columns a tile
(128 and 448 k a half), a last tile partly filled, images shared by two tiles, FP16 and BF16, one class without a
third of its directions."""
import numpy as np
import pytest

from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,coarse,n,holes", [("fp16", 16, 1250, False), ("bf16", 18, 1251, True),
                                                      ("fp16", 32, 1280, True)])
def test_resident_columns_match_tiles(engine, precision, coarse, n, holes):
    print(f"[pq cols {precision} coarse={coarse} n={n} holes={holes}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=coarse, K=1, order=2, offset_range=5.0,
                                        n=n, snr=0.5, seed=3)
    if holes:
        pd = np.asarray(prob["pdf_direction"], float).reshape(1, -1)
        pd[:, ::3] = 0
        prob["pdf_direction"] = (pd / pd.sum()).reshape(np.shape(prob["pdf_direction"]))
    synth.load_engine(engine, prob, precision=precision)
    out = {}
    for mode in ("full", "list"):
        engine.set_coarse_mode(mode)
        engine.reset_sums()
        r = engine.expectation(batch)
        out[mode] = (r, engine.get_sums())
    st = engine.coarse_stats()
    print("  list_max", st["list_max"], "total", st["list_total"], flush=True)
    engine.set_coarse_mode("list")
    assert 0 < st["list_total"] and st["mode"] == 0
    (rf, sf), (r, s) = out["full"], out["list"]
    for k in ("argmax", "nr_sign", "min_diff2", "min_diff2_coarse"):
        np.testing.assert_array_equal(r[k], rf[k], err_msg=k)
    for k in ("sum_weight_coarse", "sum_weight", "sig_weight_coarse", "sig_weight"):
        np.testing.assert_allclose(r[k], rf[k], rtol=1e-11, err_msg=k)
    for k in ("wsum_pdf_class", "wsum_sigma2_noise", "wsum_scalars"):
        np.testing.assert_allclose(s[k], sf[k], rtol=1e-10, err_msg=k)
