"""Results of several MB reach the host through a ring of pinned slots, smaller ones by a plain copy: the same pool
prepared at once (7.6 MB, the last piece partly filled), and a size that takes many turns of the ring (42 MB), must be
byte for byte what its images give a few at a time (the power spectra, which travel with them, are sums of up to 400
non-negative terms in the order the atomics happen to take: equal to 400 roundings)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b, k):
    np.testing.assert_allclose(a, b, rtol=400 * 2.0 ** -53 if k == "power_img" else 0, atol=0, err_msg=k)


@pytest.mark.parametrize("n,ori,cur", [(71, 100, 72), (129, 128, 126)])
def test_large_results_match_small_ones(engine, n, ori, cur):
    engine.configure(ref_dim=3, ori_size=ori, current_size=cur, coarse_size=cur, nr_classes=1, nr_groups=1,
                     adaptive_oversampling=0, nr_dir=12, nr_psi=6, nr_trans=1, adaptive_fraction=0.999,
                     sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0, do_ctf_correction=1,
                     refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)
    rng = np.random.default_rng(n)
    img = rng.normal(size=(n, ori, ori))
    off = rng.uniform(-4, 4, (2, n))
    ctf = np.column_stack([rng.uniform(1e4, 3e4, (n, 2)), rng.uniform(0, 180, n), np.full(n, 300.0), np.full(n, 2.7),
                           np.full(n, 0.1), np.zeros(n)])
    kw = dict(pixel_size=1.5, particle_diameter=100.0)
    whole = engine.prepare_images(img, off[0], off[1], ctf=ctf, **kw)
    again = engine.prepare_images(img, off[0], off[1], ctf=ctf, **kw)
    for i in range(0, n, 10):
        part = engine.prepare_images(img[i:i + 10], off[0, i:i + 10], off[1, i:i + 10], ctf=ctf[i:i + 10], **kw)
        for k, v in part.items():
            same(whole[k][i:i + 10], v, k)
    for k, v in whole.items():
        same(v, again[k], k)
