"""Whole 2D images (rome_backproject_images) at once: many images of one class are spread over the chip, not summed by one
block.  6000 images of 32^2 take no longer than 1.5 times what the same images take in 3D, whose bricks are spread
(one block for all of them: twice as long), and their grid is the sum of the images' own (each added alone, FP32
sums of 6000 terms of one sign a grid point at most in another order: 1e-4 of the largest)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _configure(engine, dim):
    engine.configure(ref_dim=dim, ori_size=32, current_size=32, coarse_size=32, nr_classes=1, nr_groups=1,
                     adaptive_oversampling=0, nr_dir=12 if dim == 3 else 1, nr_psi=6, nr_trans=1,
                     adaptive_fraction=0.999, sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0,
                     do_ctf_correction=1, refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)


def test_many_images(engine):
    rng = np.random.default_rng(3)
    n, F2 = 6000, 32 * 17
    im = dict(fnomask_re=rng.normal(size=(n, F2)), fnomask_im=rng.normal(size=(n, F2)), fctf=rng.uniform(0.2, 1, (n, F2)))
    euler = np.zeros((n, 3))
    euler[:, 2] = rng.uniform(0, 360, n)
    shift = rng.uniform(-2, 2, (n, 2))
    ms = {}
    for dim in (3, 2):
        _configure(engine, dim)
        t = []
        for _ in range(6):
            engine.reset_sums()
            t0 = time.perf_counter()
            engine.backproject_images(0, im, euler, shift)
            t.append(1e3 * (time.perf_counter() - t0))
        ms[dim] = float(np.median(t[1:]))
    print("[bp images 2d] ms by dimension", ms, flush=True)
    data, weight = engine.get_backprojector(0)
    part_d, part_w = np.zeros_like(data), np.zeros_like(weight)
    for a in range(0, n, 750):
        engine.reset_sums()
        engine.backproject_images(0, {k: v[a:a + 750] for k, v in im.items()}, euler[a:a + 750], shift[a:a + 750])
        d, w = engine.get_backprojector(0)
        part_d, part_w = part_d + d, part_w + w
    assert np.max(np.abs(weight - part_w)) <= 1e-4 * np.max(part_w)
    assert np.max(np.abs(data - part_d)) <= 1e-4 * np.max(part_w)
    assert ms[2] <= 1.5 * ms[3]
