"""The gridding iterations of rome_reconstruct (dense FP64 transforms in tiles of 16 rows) at the sizes where a
tile, a wave's share of tiles or the blob's end changes: H = current_size + 2 of 16, 18, 32, 34, 48, 50 and 66
rows in 3D, up to 202 in 2D, with current_size = ori_size (the blob table ends inside the grid) and below.

Both sides are FP64.  A dense sum of at most 2 H = 404 terms is off by less than 404 * 2^-53 = 5e-14 of its
terms' sum; five such stages in each of 10 iterations, the weights divided by values of order 1, stay below
50 * 5e-14 = 3e-12: the maps are held to 1e-10 of their largest value."""
import numpy as np
import pytest

import oracle.mstep as OM

pytestmark = pytest.mark.gpu


def _grids(rng, dim, cur):
    P = 2 * (2 * (cur // 2) + 1) + 1
    shape = (P, P, P // 2 + 1) if dim == 3 else (P, P // 2 + 1)
    idx = np.indices(shape)
    r2 = sum((idx[a] - P // 2) ** 2 for a in range(dim - 1)) + idx[-1] ** 2
    inside = r2 <= (2 * (cur // 2)) ** 2
    data = (rng.normal(size=shape) + 1j * rng.normal(size=shape)) * inside / (1.0 + np.sqrt(r2))
    weight = rng.uniform(0.5, 2.0, shape) * inside
    weight[rng.random(shape) < 0.1] = 0.0  # voxels no slice reached
    return data, weight


@pytest.mark.parametrize("dim,ori,cur", [(3, 14, 14), (3, 16, 16), (3, 30, 30), (3, 40, 32), (3, 46, 46), (3, 52, 48),
                                         (3, 64, 64), (2, 2, 2), (2, 14, 14), (2, 20, 16), (2, 96, 94), (2, 126, 126),
                                         (2, 160, 128), (2, 200, 200), (2, 210, 200)])
def test_gridding_sizes(engine, dim, ori, cur):
    print(f"[gridding dim={dim} ori={ori} cur={cur}]", flush=True)
    engine.configure(ref_dim=dim, ori_size=ori, current_size=cur, coarse_size=cur, nr_classes=1, nr_groups=1,
                     adaptive_oversampling=0, nr_dir=12 if dim == 3 else 1, nr_psi=6, nr_trans=1,
                     adaptive_fraction=0.999, sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0,
                     do_ctf_correction=1, refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)
    rng = np.random.default_rng(100 * cur + dim)
    data, weight = _grids(rng, dim, cur)
    tau2 = rng.uniform(0.5, 2.0, ori // 2 + 1)
    for iters, do_map in ((10, True), (1, False)):
        kw = dict(max_iter_preweight=iters, do_map=do_map, minres_map=5, tau2_fudge=1.0, normalise=1.0)
        got = engine.reconstruct(0, tau2, data=data, weight=weight, **kw)
        want = OM.reconstruct(data, weight, ori, cur, tau2=tau2, **kw)
        scale = np.max(np.abs(want[0]))
        assert np.all(np.isfinite(got[0])) and np.max(np.abs(got[0] - want[0])) <= 1e-10 * scale, (iters, do_map)
        np.testing.assert_allclose(got[2], want[2], rtol=1e-10)
        np.testing.assert_allclose(got[3], want[3], rtol=1e-10)
