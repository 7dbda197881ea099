"""The gridding iterations where their form changes: 2D sizes on both sides of the split into one-wave blocks (7 row tiles of
16 with the blob table ended inside the grid, 5 without), the largest current_size that rome_configure accepts (H = 204 of
the 240 rows the transforms take; 204 is refused), and in 3D more than 128 rows without the table's end (more than 64 KB
of LDS a block).  Bars as for the other sizes: dense FP64 sums of at most 408 terms, 1e-10 of the largest value."""
import numpy as np
import pytest

import oracle.mstep as OM
from test_gpu_gridding import _grids

pytestmark = pytest.mark.gpu


def _configure(engine, dim, ori, cur):
    engine.configure(ref_dim=dim, ori_size=ori, current_size=cur, coarse_size=cur, nr_classes=1, nr_groups=1,
                     adaptive_oversampling=0, nr_dir=12 if dim == 3 else 1, nr_psi=6, nr_trans=1,
                     adaptive_fraction=0.999, sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0,
                     do_ctf_correction=1, refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)


@pytest.mark.parametrize("dim,ori,cur,iters", [(2, 94, 94, 10), (2, 98, 98, 10), (2, 100, 62, 10), (2, 100, 64, 10),
                                               (2, 98, 78, 3), (2, 202, 202, 10), (2, 300, 202, 10), (3, 140, 128, 1)])
def test_gridding_forms(engine, dim, ori, cur, iters):
    print(f"[gridding forms dim={dim} ori={ori} cur={cur}]", flush=True)
    _configure(engine, dim, ori, cur)
    rng = np.random.default_rng(100 * cur + dim)
    data, weight = _grids(rng, dim, cur)
    tau2 = rng.uniform(0.5, 2.0, ori // 2 + 1)
    kw = dict(max_iter_preweight=iters, do_map=iters > 1, minres_map=5, tau2_fudge=1.0, normalise=1.0)
    got = engine.reconstruct(0, tau2, data=data, weight=weight, **kw)
    want = OM.reconstruct(data, weight, ori, cur, tau2=tau2, **kw)
    scale = np.max(np.abs(want[0]))
    assert np.all(np.isfinite(got[0])) and np.max(np.abs(got[0] - want[0])) <= 1e-10 * scale
    np.testing.assert_allclose(got[2], want[2], rtol=1e-10)
    np.testing.assert_allclose(got[3], want[3], rtol=1e-10)


def test_larger_sizes_are_refused(engine):
    with pytest.raises(Exception, match="current_size too large"):
        _configure(engine, 2, 256, 204)
