"""rome_backproject_images (binned scatter in 3D, bands in 2D) against the FP64 oracle's backprojection: one
image, a pool past the 1024 images of one device pass, with and without CTF images, into the second of two classes
and on top of an earlier call.  Corner weights and values are FP32 products of a few terms (a few 2^-24 each) and a
voxel's sum takes at most a few thousand of them: 1e-5 relative L2, as for the E-step's grids."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,ori,cur,n,ctf", [(3, 16, 16, 1, True), (3, 24, 18, 70, True), (3, 16, 16, 1100, False),
                                               (3, 56, 56, 40, True), (2, 16, 16, 1, True), (2, 24, 18, 70, False), (2, 20, 20, 1100, True), (2, 100, 100, 9, True)])
def test_backproject_images(engine, dim, ori, cur, n, ctf):
    print(f"[bp images dim={dim} ori={ori} cur={cur} n={n} ctf={ctf}]", flush=True)
    engine.configure(ref_dim=dim, ori_size=ori, current_size=cur, coarse_size=cur, nr_classes=2, nr_groups=1,
                     adaptive_oversampling=0, nr_dir=12 if dim == 3 else 1, nr_psi=6, nr_trans=1,
                     adaptive_fraction=0.999, sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0,
                     do_ctf_correction=1, refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)
    engine.reset_sums()
    rng = np.random.default_rng(n + dim)
    F2 = cur * (cur // 2 + 1)
    F = (rng.normal(size=(n, F2)) + 1j * rng.normal(size=(n, F2))).astype(np.complex64).astype(np.complex128)
    c = rng.uniform(-1, 1, (n, F2)).astype(np.float32).astype(np.float64)
    c[:, 3] = 0.0  # no weight: no contribution
    euler = np.column_stack([rng.uniform(-180, 180, n), rng.uniform(0, 180, n), rng.uniform(0, 360, n)])
    shift = rng.uniform(-3, 3, (n, 2))
    img = dict(fnomask_re=F.real, fnomask_im=F.imag, fctf=c if ctf else None)
    cut = n // 3  # two calls add up
    for a, b in ((0, cut), (cut, n)):
        sub = {k: None if v is None else v[a:b] for k, v in img.items()}
        engine.backproject_images(1, sub, euler[a:b], shift[a:b])
    pad = O.pad_size(cur, ori)
    gn = pad * pad * (pad // 2 + 1) if dim == 3 else pad * (pad // 2 + 1)
    data, weight = np.zeros(2 * gn), np.zeros(gn)
    keep = np.where(O.mresol(cur) >= 0, 1.0, 0.0)
    for i in range(n):
        sr, si = O.shift_image(F[i].real, F[i].imag, cur, shift[i, 0], shift[i, 1], ori)
        w = (c[i] if ctf else np.ones(F2)) * keep
        A = O.euler_matrix(*euler[i]) if dim == 3 else O.euler_matrix(0, 0, euler[i, 2])
        (O.backproject3d if dim == 3 else O.backrotate2d)(data, weight, pad, cur // 2, A, cur, sr * w, si * w, w * w)
    dg, wg = engine.get_backprojector(1)
    assert np.linalg.norm(dg - data) <= 1e-5 * np.linalg.norm(data)
    assert np.linalg.norm(wg - weight) <= 1e-5 * np.linalg.norm(weight)
    d0, w0 = engine.get_backprojector(0)
    assert not d0.any() and not w0.any()
