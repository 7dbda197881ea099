"""The window of a padded transform into the projector grid at row lengths around a wave (33, 66 and 133 elements, 2D
and 3D, the ball cut or complete): grid and spectrum against the FP64 oracle to 1e-12 / 1e-10 of their scale (both are
FP64 transforms of the same samples), zeros outside the ball exact, also over what an earlier map left there, and the
FP32 grid, seen through a projection, the same without the FP64 one."""
import numpy as np
import pytest

import oracle.mstep as OM
from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,ori,cur", [(3, 30, 30), (3, 64, 64), (3, 64, 22), (2, 130, 130), (2, 130, 60)])
def test_window_covers_the_grid(engine, dim, ori, cur):
    engine.configure(ref_dim=dim, ori_size=ori, current_size=cur, coarse_size=cur, nr_classes=1, nr_groups=1,
                     adaptive_oversampling=0, nr_dir=12 if dim == 3 else 1, nr_psi=6, nr_trans=1, adaptive_fraction=0.999,
                     sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0, do_ctf_correction=1,
                     refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)
    rng = np.random.default_rng(ori + cur)
    engine.fourier_map(0, 100 * rng.normal(size=(ori,) * dim))
    vol = synth.blob_volume(ori, 12, (1.5, 3.0), 0.35 * ori, rng, ndim=dim)
    ps, _, grid = engine.fourier_map(0, vol)
    g_ref, p_ref, _ = OM.fourier_map(vol, cur)
    assert grid.shape == g_ref.shape
    assert np.max(np.abs(grid - g_ref)) <= 1e-12 * np.max(np.abs(g_ref))
    assert np.all(grid[g_ref == 0] == 0)
    np.testing.assert_allclose(ps, p_ref, rtol=1e-10, atol=1e-14 * p_ref.max())
    A = np.stack([np.eye(3)] + [synth.euler_matrix(*rng.uniform([-180, 0, 0], [180, 180, 360])) for _ in range(3)])
    seen = engine.project(0, cur, A)
    engine.fourier_map(0, 100 * rng.normal(size=(ori,) * dim), want_grid=False)
    engine.fourier_map(0, vol, want_grid=False)
    for a, b in zip(seen, engine.project(0, cur, A)):
        np.testing.assert_array_equal(a, b)
