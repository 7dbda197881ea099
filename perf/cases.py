"""The work that users of this engine have it do, as cases for timing and for comparing results.

A case is a dict of plain values; its "kind" names the call:

  pool   one pool of particle images through the E-step (rome_expectation_device) and its sums; 3D and 2D,
         with and without oversampling, in the three arithmetic arms of the coarse cross term
  fine   the fine pass of a pool whose coarse significance is given (rome_expectation_fine_device)
  iter   one iteration: pools, model update, every class reconstructed
  prep   image preparation of a pool of real-space images on the host (rome_prepare_images)
  recon  a class map from its backprojection grids (rome_reconstruct)
  fmap   the projector grid of a class map (rome_fourier_map)
  offl   offline reconstruction: images at known poses backprojected, then the map
  train  the learned pose proposal trained on collected posteriors

Inputs are synthetic: maps of Gaussian blobs, particles = CTF * projection * shift + white noise at a
given SNR, made here with torch in 64 bits from the seed alone.  exact() restates each call in 64 bits.
"""
import math

import numpy as np
import torch

import rome_amd
from rome_amd import PRECISIONS, Engine

DEV = "cuda"
F64 = torch.float64
C128 = torch.complex128
PI = math.pi


# ------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the plain 3D classification at its usual size, a large pool, FP16 cross term: the headline workload
        _pool("pool3d_128_fp16", prec="fp16", n=2000),
        # the same search in the default arithmetic; a pool of ordinary size
        _pool("pool3d_128_fp32", prec="fp32", n=250),
        # early iteration at a box and a resolution off the powers of two, three optics groups, odd pool
        _pool("pool3d_100_bf16", prec="bf16", n=333, ori=100, cur=72, coarse=20, K=3, rng=3.0, groups=3, snr=0.08),
        # a few particles of a small box (a live preview, the tail of a dataset): latency and launches
        _pool("pool3d_32_small", prec="fp32", n=5, ori=32, cur=32, coarse=16, K=2, order=1, rng=2.0, snr=0.5),
        # 2D classification of 64^2 particles, 36 angles x 29 shifts, one pass, broad posteriors
        _pool("pool2d_64", prec="fp32", n=1000, ori=64, cur=64, coarse=64, K=10, dim=2, psi=10.0, rng=3.0, over=0, snr=0.05),
        # late iteration of a large box: the search is local, its samples come from the pass before
        dict(name="fine3d_192", kind="fine", n=100, ori=192, cur=192, coarse=48, K=2, order=3, rng=4.0, dim=3, over=1,
             prec="fp32", groups=1, snr=0.05, median=300, psi=0.0),
        # one iteration of a 2D classification with adaptive oversampling and a partial resolution
        dict(_pool("iter2d_64", prec="fp32", n=400, ori=64, cur=48, coarse=24, K=10, dim=2, psi=10.0, rng=3.0, over=1, snr=0.1),
             kind="iter", pools=2),
        # what every particle goes through before its first E-step of an iteration
        dict(name="prep_128", kind="prep", n=500, ori=128, cur=96, ctf=1, norm=1, noise=0),
        # the M-step of a class: a 128^3 map from its grids, with the MAP term
        dict(name="recon3d_128", kind="recon", ori=128, cur=128, dim=3, views=400, do_map=1, iters=10),
        # a new 192^3 class map made a reference
        dict(name="fmap3d_192", kind="fmap", ori=192, cur=192, dim=3),
        # the offline tool: particles with known poses to a map of an odd-sized grid
        dict(name="offl3d_100", kind="offl", n=400, ori=100, cur=100, dim=3, ctf=1),
        # the proposal network of a small search trained on one pool's posteriors
        dict(_pool("train_64", prec="fp16", n=1024, ori=64, cur=64, coarse=24, K=2, rng=2.0, snr=0.5), kind="train",
             hidden=1024, coef=812, batch=256, epochs=8, lr=1e-3),
    ]


def _pool(name, prec, n, ori=128, cur=128, coarse=24, K=4, order=2, rng=5.0, dim=3, over=1, groups=1, snr=0.05, psi=0.0):
    return dict(name=name, kind="pool", prec=prec, n=n, ori=ori, cur=cur, coarse=coarse, K=K, order=order, rng=rng, dim=dim,
                over=over, groups=groups, snr=snr, psi=psi)


def _log(r, lo, hi):
    return lo * (hi / lo) ** r.random()


def _even(v):
    return 2 * int(round(v / 2))


def draw(rng):
    r = rng
    kind = r.choice(["pool3", "pool3", "pool3", "pool2", "pool2", "fine", "iter", "prep", "recon", "fmap", "offl", "train"])
    ori = _even(_log(r, 32, 128))
    cur = ori if r.random() < 0.5 else _even(r.uniform(0.6, 1.0) * ori)
    snr = round(min(0.6, 0.05 * (128 / ori) ** 1.66 * r.uniform(1, 2)), 3)
    coarse = min(cur, _even(r.uniform(16, 28)))
    if kind in ("pool3", "train"):
        order, K = r.choice([1, 2, 2]), r.choice([1, 2, 3, 4, 5])
        t = r.choice([2.0, 3.0, 4.0, 5.0])
        n = int(_log(r, 3, 1500 if order == 2 else 2000)) if kind == "pool3" else 32 * r.randint(12, 40)
        c = _pool("", r.choice(["fp32", "bf16", "fp16"]), n, ori, cur, coarse, K, order, t, 3, 1, r.choice([1, 1, 2, 5]), snr)
        if kind == "train":
            ori = min(ori, 96)
            c.update(kind="train", ori=ori, cur=ori, coarse=min(coarse, 24), K=r.choice([1, 2]), order=2, rng=2.0, groups=1,
                     prec=r.choice(["bf16", "fp16"]), snr=0.5, hidden=r.choice([512, 1024]), coef=r.choice([200, 406]),
                     batch=32 * r.randint(2, 12), epochs=r.choice([4, 8]), lr=1e-3)
        c.pop("name")
        return c
    if kind in ("pool2", "iter"):
        dim = 2 if kind == "pool2" else r.choice([2, 2, 3])
        over = 1 if dim == 3 else r.choice([0, 1])
        if kind == "iter":
            ori = min(ori, 96) if dim == 2 else min(ori, 72)
            cur = min(cur, ori)
        snr = round(min(0.6, 0.05 * (128 / ori) ** 1.66 * r.uniform(1, 2)), 3)
        c = _pool("", r.choice(["fp32", "fp32", "fp16"]) if over else "fp32", int(_log(r, 5, 1200 if kind == "pool2" else 300)),
                  ori, cur, min(coarse, cur) if over else cur, r.randint(1, 20) if dim == 2 else r.randint(1, 3),
                  1 if dim == 3 else 0, r.choice([2.0, 3.0]), dim, over, r.choice([1, 3]), snr,
                  r.choice([5.0, 7.5, 10.0]) if dim == 2 else 0.0)
        if kind == "iter":
            c.update(kind="iter", pools=r.randint(1, 3))
        c.pop("name")
        return c
    if kind == "fine":
        ori = _even(_log(r, 64, 192))
        cur = ori if r.random() < 0.5 else _even(r.uniform(0.7, 1.0) * ori)
        return dict(kind="fine", n=int(_log(r, 5, 100)), ori=ori, cur=cur, coarse=min(cur, 48), K=r.randint(1, 3), order=r.choice([2, 3]),
                    rng=r.choice([3.0, 4.0, 5.0]), dim=3, over=1, prec="fp32", groups=r.choice([1, 2]), snr=snr,
                    median=int(_log(r, 10, 300)), psi=0.0)
    if kind == "prep":
        return dict(kind="prep", n=int(_log(r, 4, 500)), ori=ori, cur=cur, ctf=r.choice([0, 1, 1]), norm=r.choice([0, 1]),
                    noise=r.choice([0, 0, 1]))
    dim = r.choice([2, 3, 3])
    if kind == "recon":
        return dict(kind="recon", ori=ori, cur=cur, dim=dim, views=int(_log(r, 50, 400)), do_map=r.choice([0, 1, 1]),
                    iters=r.choice([5, 10, 10]))
    if kind == "fmap":
        ori = _even(_log(r, 32, 192))
        return dict(kind="fmap", ori=ori, cur=_even(ori * r.choice([1.0, 1.0, 0.6, 0.8])), dim=dim)
    return dict(kind="offl", n=int(_log(r, 10, 500)), ori=ori, cur=ori, dim=dim, ctf=r.choice([0, 1, 1]))


# ------------------------------------------------------------------------------------- geometry and maps
def _half_xy(size):
    F = size // 2 + 1
    i = torch.arange(size)
    y = torch.where(i < F, i, i - size)[:, None].expand(size, F).reshape(-1)
    x = torch.arange(F)[None, :].expand(size, F).reshape(-1)
    return x.to(DEV), y.to(DEV)


def _shell(size):
    """Shell of each half-plane pixel (rounded radius; -1: outside, or the x = 0 column counted twice)."""
    x, y = _half_xy(size)
    r = torch.floor(torch.sqrt((x * x + y * y).to(F64)) + 0.5).long()
    return torch.where((r < size // 2 + 1) & ~((x == 0) & (y < 0)), r, torch.full_like(r, -1))


def _signed(n, half):
    k = torch.arange(n, device=DEV)
    return torch.where(k < half, k, k - n)


def _rad2(*axes):
    out = 0
    for d, a in enumerate(axes):
        shape = [1] * len(axes)
        shape[d] = -1
        out = out + (a * a).reshape(shape)
    return out


def _pad(cur):
    return 2 * (2 * (cur // 2) + 1) + 1


def _matrices(euler):
    """[.., 3] rot, tilt, psi in degrees -> [.., 3, 3]."""
    a, b, g = (torch.deg2rad(torch.as_tensor(euler, dtype=F64, device=DEV)[..., i]) for i in range(3))
    ca, cb, cg, sa, sb, sg = a.cos(), b.cos(), g.cos(), a.sin(), b.sin(), g.sin()
    cc, cs, sc, ss = cb * ca, cb * sa, sb * ca, sb * sa
    m = [cg * cc - sg * sa, cg * cs + sg * ca, -cg * sb, -sg * cc - cg * sa, -sg * cs + cg * ca, sg * sb, sc, ss, cb]
    return torch.stack(m, -1).reshape(*a.shape, 3, 3)


def _blobs(ori, dim, count, gen):
    """A map of Gaussian blobs inside a sphere of 0.39 ori (64 bits; separable)."""
    c = torch.randn(count, dim, generator=gen, dtype=F64)
    c = c / c.norm(dim=1, keepdim=True) * (0.39 * ori * torch.rand(count, 1, generator=gen, dtype=F64) ** (1 / dim))
    s = (0.016 + 0.03 * torch.rand(count, 1, generator=gen, dtype=F64)) * ori + 0.5
    amp = 0.5 + torch.rand(count, generator=gen, dtype=F64)
    ax = torch.arange(ori, dtype=F64)[None, :] - ori // 2
    g = [torch.exp(-((ax - c[:, d : d + 1]) ** 2) / (2 * s * s)).to(DEV) for d in range(dim)]
    amp = amp.to(DEV)
    if dim == 2:
        return (g[0] * amp[:, None]).T @ g[1]
    yx = (g[1][:, :, None] * g[2][:, None, :]).reshape(count, -1)
    return ((g[0] * amp[:, None]).T @ yx).reshape(ori, ori, ori)


def _radius(ori, dim):
    a = (torch.arange(ori, device=DEV) - ori // 2).to(F64)
    return torch.sqrt(_rad2(*([a] * dim)))


def _sinc2(ori, dim):
    q = PI * _radius(ori, dim) / (2 * ori)
    return torch.where(q > 0, (torch.sin(q) / torch.where(q > 0, q, torch.ones_like(q))) ** 2, torch.ones_like(q))


def _fourier_map(vol, cur, spectrum=False):
    """The projector grid of computeFourierTransformMap (and the power spectrum and gridding-corrected map)."""
    dim, ori = vol.dim(), vol.shape[0]
    r_max, N = min(cur, ori) // 2, 2 * ori
    corr = vol / _sinc2(ori, dim)
    P = torch.zeros((N,) * dim, dtype=F64, device=DEV)
    P[(slice(N // 2 - ori // 2, N // 2 - ori // 2 + ori),) * dim] = corr
    F = torch.fft.rfftn(torch.roll(P, (N // 2,) * dim, tuple(range(dim)))) * ((8.0 * ori if dim == 3 else 4.0) / N**dim)
    pad = _pad(cur)
    k = torch.arange(pad, device=DEV) - pad // 2
    half = torch.arange(pad // 2 + 1, device=DEV)
    keep = _rad2(*([torch.where(k > -(N // 2), k, k * 4)] * (dim - 1)), half)  # -N/2 is there as +N/2 only
    idx = k % N
    half = half.clamp(max=N // 2)
    sel = keep <= 4 * r_max * r_max
    G = F[idx][:, idx][:, :, half] if dim == 3 else F[idx][:, half]
    G = torch.where(sel, G, torch.zeros_like(G))
    if not spectrum:
        return G
    sh = torch.floor(torch.sqrt(keep[sel].to(F64)) / 2 + 0.5).long()
    pw, ct = _shell_sums(sh, G[sel].abs() ** 2 / 2, ori), _shell_sums(sh, torch.ones_like(sh, dtype=F64), ori)
    return G, torch.where(ct < 1, torch.zeros_like(pw), pw / ct.clamp(min=1)), corr


def _shell_sums(sh, v, ori):
    return torch.tensor(np.bincount(sh.cpu().numpy(), v.cpu().numpy(), ori // 2 + 1), device=DEV)


def _corners(A, x, y, pad):
    """Flat grid indices [rot][pix][2^dim] and weights of the trilinear samples, and which are mirrored."""
    padF, c = pad // 2 + 1, pad // 2
    dim = 3 if A.shape[-1] == 3 else 2
    p = 2 * (A[:, 0, :, None] * x[None, None, :].to(F64) + A[:, 1, :, None] * y[None, None, :].to(F64))  # [rot][axis][pix]
    neg = p[:, 0] < 0
    p = torch.where(neg[:, None], -p, p)
    f = torch.floor(p)
    w1 = p - f
    i0 = f.long()
    i0[:, 1:] += c
    idx, wgt = [], []
    for q in range(2**dim):
        d = [(q >> a) & 1 for a in range(dim)]
        w = 1
        for a in range(dim):
            w = w * (w1[:, a] if d[a] else 1 - w1[:, a])
        i = (i0[:, 1] + d[1]) * padF + i0[:, 0] + d[0]
        if dim == 3:
            i = i + (i0[:, 2] + d[2]) * (pad * padF)
        idx.append(i)
        wgt.append(w)
    return torch.stack(idx, -1), torch.stack(wgt, -1), neg


def _project(grid, A, x, y, r2max, chunk=64):
    """Slices [rot][pix] of a projector grid, 64 bits."""
    pad = grid.shape[0]
    flat = grid.reshape(-1)
    inside = (x * x + y * y) <= r2max
    xi, yi = x * inside, y * inside
    out = []
    A = A if grid.dim() == 3 else A[:, :2, :2]
    for a in A.split(chunk):
        idx, w, neg = _corners(a, xi, yi, pad)
        v = (flat[idx] * w).sum(-1)
        out.append(torch.where(neg, v.conj(), v) * inside)
    return torch.cat(out)


def _phase(sx, sy, x, y, ori):
    """Tabulated shift phases [shift][pix] (shiftImageInFourierTransform's 5000-entry table, floor-indexed)."""
    xs = (sx / -float(ori))[:, None]
    ys = (sy / -float(ori))[:, None]
    dot = 2 * PI * (x[None, :].to(F64) * xs + y[None, :].to(F64) * ys)
    it = (dot.abs() / (2 * PI / 5000.0)).long() % 5000
    ang = it.to(F64) * (2 * PI / 5000.0)
    s = torch.where(dot < 0, -ang.sin(), ang.sin())
    ident = (xs.abs() < 1e-6) & (ys.abs() < 1e-6)
    return torch.where(ident, torch.ones_like(dot, dtype=C128), torch.complex(ang.cos(), s))


def _ctf(size, ori, angpix, par):
    """CTF images [n][pix] of defocus U, V, angle, 300 kV, Cs 2.7, Q0 0.1 (par [n][7])."""
    x, y = _half_xy(size)
    X, Y = x.to(F64) / (ori * angpix), y.to(F64) / (ori * angpix)
    u2 = X * X + Y * Y
    kv, cs, q0 = par[:, 3:4] * 1e3, par[:, 4:5] * 1e7, par[:, 5:6]
    lam = 12.2643247 / torch.sqrt(kv * (1.0 + kv * 0.978466e-6))
    ang = torch.atan2(Y, X)[None] - par[:, 2:3] * PI / 180
    defoc = -(par[:, 0:1] + par[:, 1:2]) / 2 - (par[:, 0:1] - par[:, 1:2]) / 2 * torch.cos(2 * ang)
    defoc = torch.where((X.abs() < 1e-6) & (Y.abs() < 1e-6), torch.zeros_like(defoc), defoc)
    arg = PI * lam * defoc * u2 + PI / 2 * cs * lam**3 * u2 * u2
    return -(torch.sqrt(1 - q0 * q0) * arg.sin() - q0 * arg.cos()) * torch.exp(-par[:, 6:7] / 4 * u2)


def _ctf_par(n, gen):
    u = torch.rand(n, 3, generator=gen, dtype=F64)
    p = torch.empty(n, 7, dtype=F64)
    p[:, 0], p[:, 1], p[:, 2] = 1e4 + 2e4 * u[:, 0], 1e4 + 2e4 * u[:, 1], 180 * u[:, 2]
    p[:, 3:] = torch.tensor([300.0, 2.7, 0.1, 0.0], dtype=F64)
    return p.to(DEV)


def _poses(n, dim, gen):
    u = torch.rand(n, 3, generator=gen, dtype=F64)
    e = torch.stack([360 * u[:, 0] - 180, torch.rad2deg(torch.acos(2 * u[:, 1] - 1)), 360 * u[:, 2]], 1)
    if dim == 2:
        e[:, :2] = 0
    return e.to(DEV)


# ------------------------------------------------------------------------------------------ E-step inputs
def _search(case):
    """Sampling tables (as the caller's sampler gives them, perturbed) and the sizes that follow."""
    d3, over = case["dim"] == 3, case["over"]
    pert = 0.25
    if d3:
        pc = rome_amd.pose_table3d(case["order"], 0, pert)
        pf = rome_amd.pose_table3d(case["order"], 1, pert) if over else None
        D, PSI = pc.shape[:2]
    else:
        pc = rome_amd.pose_table2d(case["psi"], 0, pert)
        pf = rome_amd.pose_table2d(case["psi"], 1, pert) if over else None
        D, PSI = 1, len(pc)
    tx, ty = rome_amd.translations(case["rng"], 1.0)
    scx, scy = rome_amd.shift_table(case["rng"], 1.0, 0, pert)
    sfx, sfy = rome_amd.shift_table(case["rng"], 1.0, 1, pert) if over else (None, None)
    return dict(pose_coarse=pc, pose_fine=pf, shift_coarse_x=scx[:, 0], shift_coarse_y=scy[:, 0], shift_fine_x=sfx,
                shift_fine_y=sfy, trans_x=tx, trans_y=ty), D, PSI, len(tx)


def _data(case, seed):
    """Maps, model and images of a pool (or of all pools of an iteration), on the GPU."""
    gen = torch.Generator().manual_seed(int(seed) * 2 + 1)
    K, ori, cur, dim, G = case["K"], case["ori"], case["cur"], case["dim"], case["groups"]
    n = case["n"] * case.get("pools", 1)
    tables, D, PSI, T = _search(case)
    grids = torch.stack([_fourier_map(_blobs(ori, dim, 200 if ori >= 64 else 60, gen), cur) for _ in range(K)])
    x, y = _half_xy(cur)
    cls = torch.randint(K, (n,), generator=gen)
    euler, par = _poses(n, dim, gen), _ctf_par(n, gen)
    off = torch.randint(-2, 3, (2, n), generator=gen).to(F64).to(DEV)
    shift = ((2 * torch.rand(n, 2, generator=gen, dtype=F64) - 1) * (case["rng"] - 0.5)).to(DEV)
    ctf = torch.cat([_ctf(cur, ori, 1.5 * 128 / ori, p) for p in par.split(256)]).float()
    F = torch.empty(n, x.numel(), dtype=torch.complex64, device=DEV)
    A = _matrices(euler)
    for k in range(K):
        sel = torch.nonzero(cls == k)[:, 0].to(DEV)
        if len(sel):
            F[sel] = _project(grids[k], A[sel], x, y, (cur // 2) ** 2).to(torch.complex64)
    for q in range(0, n, 256):
        ph = 2 * PI * (x[None].to(F64) * shift[q : q + 256, :1] + y[None].to(F64) * shift[q : q + 256, 1:]) / ori
        F[q : q + 256] *= (ctf[q : q + 256] * torch.polar(torch.ones_like(ph), ph)).to(torch.complex64)
    inside = (x * x + y * y) <= (cur // 2) ** 2
    sigma2 = 0.5 * float((F[:, inside].abs().double() ** 2).mean()) / case["snr"]
    gd = torch.Generator(device=DEV).manual_seed(int(seed) + 7)
    F += torch.view_as_complex(torch.randn(n, x.numel(), 2, generator=gd, device=DEV) * math.sqrt(sigma2))
    oriF = ori // 2 + 1
    sh = _shell(ori)
    npix = torch.bincount(sh[sh >= 0], minlength=oriF).to(F64)
    power = 2 * sigma2 * npix[None] * (1 + 0.05 * torch.randn(n, oriF, generator=gd, device=DEV, dtype=F64))
    power[:, 0] = 0
    hx = power[:, cur // 2 + 1 :].sum(1).contiguous()
    if cur == ori:
        power.zero_()
    group = torch.randint(G, (n,), generator=gen, dtype=torch.int32).to(DEV)
    s2n = sigma2 * (0.9 + 0.2 * torch.rand(G, oriF, generator=gen, dtype=F64))
    pdf = 0.5 + torch.rand(K, generator=gen, dtype=F64)
    pdf = pdf / pdf.sum()
    pdir = (0.7 + 0.6 * torch.rand(K, D, generator=gen, dtype=F64)) / D * pdf[:, None]
    prior = 0.3 * torch.randn(2, K, generator=gen, dtype=F64) if dim == 2 else torch.zeros(2, K, dtype=F64)
    return dict(tables=tables, D=D, PSI=PSI, T=T, n=n, grids=grids, F=F, ctf=ctf, hx=hx, power=power, offx=off[0].contiguous(),
                offy=off[1].contiguous(), norm=(0.9 + 0.2 * torch.rand(n, generator=gen, dtype=F64)).to(DEV), group=group,
                sigma2=s2n.numpy(), pdf_class=pdf.numpy(), pdf_dir=pdir.numpy(), prior=prior.numpy(), cls=cls, euler=euler,
                shift=shift, sigma2_offset=max(1.0, (case["rng"] / 2) ** 2))


def _engine(case, d):
    e = Engine(0)
    e.configure(ref_dim=case["dim"], ori_size=case["ori"], current_size=case["cur"], coarse_size=case["coarse"],
                nr_classes=case["K"], nr_groups=case["groups"], adaptive_oversampling=case["over"], nr_dir=d["D"],
                nr_psi=d["PSI"], nr_trans=d["T"], adaptive_fraction=0.999, sigma2_fudge=1.0, sigma2_offset=d["sigma2_offset"],
                avg_norm_correction=1.0, do_ctf_correction=1, refs_are_ctf_corrected=1, do_norm_correction=1, do_map=1,
                precision=PRECISIONS[case["prec"]])
    t = d["tables"]
    e.set_sampling(t["pose_coarse"], t["pose_fine"], t["shift_coarse_x"], t["shift_coarse_y"], t["shift_fine_x"],
                   t["shift_fine_y"], t["trans_x"], t["trans_y"])
    for k in range(case["K"]):
        e.set_reference(k, torch.view_as_real(d["grids"][k]).cpu().numpy())
    e.set_model(d["sigma2"], d["pdf_class"], d["pdf_dir"], d["prior"][0], d["prior"][1])
    return e


def _ptrs(d, a, b):
    return [t[a:b].data_ptr() for t in (d["F"], d["F"], d["ctf"], d["hx"], d["power"], d["offx"], d["offy"], d["norm"], d["group"])]


def _significance(case, d, seed):
    """Lognormal numbers of coarse samples around each image's true pose: keys [n][cap], counts [n]."""
    rng = np.random.default_rng(int(seed) + 3)
    n, T, PSI, R = d["n"], d["T"], d["PSI"], d["D"] * d["PSI"]
    cnt = np.clip(np.rint(case["median"] * np.exp(rng.standard_normal(n))), 1, min(5000, R * T)).astype(np.int64)
    cap = int(cnt.max())
    Rc = _matrices(d["tables"]["pose_coarse"].reshape(-1, 3)).reshape(R, 9).float()
    Rt = _matrices(d["euler"]).reshape(n, 9).float()
    tx, ty = (torch.tensor(d["tables"][k], device=DEV).float() for k in ("trans_x", "trans_y"))
    keys = torch.full((n, cap), -1, dtype=torch.int32, device=DEV)
    for i in range(n):
        c = int(cnt[i])
        ang = torch.rad2deg(torch.arccos(((Rc @ Rt[i] - 1) / 2).clamp(-1, 1))) * (PSI / 360.0)
        a, ri = torch.topk(ang, min(R, max(16, 4 * c)), largest=False)
        far = torch.hypot(tx - d["shift"][i, 0].float(), ty - d["shift"][i, 1].float())
        q = torch.topk((a[:, None] ** 2 + far[None] ** 2).reshape(-1), c, largest=False).indices
        keys[i, :c] = ((int(d["cls"][i]) * R + ri[q // T]) * T + q % T).int()
    return keys, torch.tensor(cnt, dtype=torch.int32, device=DEV), cap


def _rotations_grid(e, case, seed):
    """Backprojection of random views into class 0, as an E-step leaves it."""
    gen = torch.Generator().manual_seed(int(seed) * 2 + 1)
    ori, cur, dim, n = case["ori"], case["cur"], case["dim"], case.get("views") or case["n"]
    x, y = _half_xy(cur)
    grid = _fourier_map(_blobs(ori, dim, 60, gen), cur)
    euler, par = _poses(n, dim, gen), _ctf_par(n, gen)
    ctf = _ctf(cur, ori, 1.5 * 128 / ori, par)
    ctf = ctf if case.get("ctf", 1) else torch.ones_like(ctf)
    F = _project(grid, _matrices(euler), x, y, (cur // 2) ** 2) * ctf
    shift = (4 * torch.rand(n, 2, generator=gen, dtype=F64) - 2).to(DEV)
    ph = 2 * PI * (x[None].to(F64) * shift[:, :1] + y[None].to(F64) * shift[:, 1:]) / ori
    F = F * torch.polar(torch.ones_like(ph), ph)
    noise = torch.randn(n, x.numel(), 2, generator=torch.Generator(device=DEV).manual_seed(int(seed) + 7), device=DEV, dtype=F64)
    F = F + torch.view_as_complex(noise) * F.abs().mean()
    # in 32 bits first: what the engine keeps of an image
    return F.to(torch.complex64).to(C128), ctf.float().double(), euler, shift


def _plain_config(case, **kw):
    c = dict(ref_dim=case.get("dim", 3), ori_size=case["ori"], current_size=case["cur"], coarse_size=case["cur"], nr_classes=1,
             nr_groups=1, adaptive_oversampling=0, nr_dir=12 if case.get("dim", 3) == 3 else 1, nr_psi=6, nr_trans=1,
             adaptive_fraction=0.999, sigma2_fudge=1.0, sigma2_offset=1.0, avg_norm_correction=1.0,
             do_ctf_correction=case.get("ctf", 1), refs_are_ctf_corrected=1, do_norm_correction=0, do_map=1, precision=0)
    c.update(kw)
    return c


def _prep_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed) + 7)
    cpu = torch.Generator().manual_seed(int(seed) * 2 + 1)
    n, ori = case["n"], case["ori"]
    vol = _blobs(ori, 2, 60, cpu)
    img = vol[None] * (0.5 + torch.rand(n, 1, 1, generator=gen, device=DEV, dtype=F64))
    img = img + torch.randn(n, ori, ori, generator=gen, device=DEV, dtype=F64) * float(vol.std()) * 3
    return dict(images=img.cpu().numpy(), xoff=(6 * torch.rand(n, generator=cpu, dtype=F64) - 3).numpy(),
                yoff=(6 * torch.rand(n, generator=cpu, dtype=F64) - 3).numpy(),
                norm=(0.8 + 0.4 * torch.rand(n, generator=cpu, dtype=F64)).numpy() if case["norm"] else None,
                ctf=_ctf_par(n, cpu).cpu().numpy() if case["ctf"] else None,
                noise=torch.randn(n, ori, ori, generator=gen, device=DEV, dtype=F64).cpu().numpy() if case["noise"] else None)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("pool", "fine", "iter", "train"):
        d = _data(case, seed)
        e = _engine(case, d)
        d["grids"] = None
        s = dict(case=case, e=e, d=d)
        if kind == "fine":
            s["keys"], s["cnt"], s["cap"] = _significance(case, d, seed)
        if kind == "train":
            e.proposal_configure(hidden=case["hidden"], nr_coef=case["coef"], max_train=case["n"], seed=int(seed))
            e.proposal_mode("collect")
            torch.cuda.synchronize()
            e.expectation_device(d["n"], *_ptrs(d, 0, d["n"]), results=False)
            e.proposal_mode("off")
        torch.cuda.synchronize()
        return s
    e = Engine(0)
    s = dict(case=case, e=e)
    if kind == "prep":
        e.configure(**_plain_config(case, do_norm_correction=case["norm"], avg_norm_correction=1.1))
        s.update(_prep_inputs(case, seed))
        n, cF, oF = case["n"], case["cur"] * (case["cur"] // 2 + 1), case["ori"] // 2 + 1
        s["dev"] = dict(fmask=torch.zeros(n, cF, 2, device=DEV), fnomask=torch.zeros(n, cF, 2, device=DEV),
                        fctf=torch.zeros(n, cF, device=DEV), highres_Xi2=torch.zeros(n, dtype=F64, device=DEV),
                        power_img=torch.zeros(n, oF, dtype=F64, device=DEV), old_offx=torch.zeros(n, dtype=F64, device=DEV),
                        old_offy=torch.zeros(n, dtype=F64, device=DEV))
    elif kind in ("recon", "offl"):
        e.configure(**_plain_config(case))
        F, ctf, euler, shift = _rotations_grid(e, case, seed)
        s["img"] = dict(fnomask_re=F.real.cpu().numpy().copy(), fnomask_im=F.imag.cpu().numpy().copy(), fctf=ctf.cpu().numpy())
        s["euler"], s["shift"] = euler.cpu().numpy(), shift.cpu().numpy()
        s["tau2"] = _tau2(case)
        if kind == "recon":
            e.reset_sums()
            e.backproject_images(0, s["img"], s["euler"], s["shift"])
    else:
        e.configure(**_plain_config(case))
        s["vol"] = _blobs(case["ori"], case["dim"], 100, torch.Generator().manual_seed(int(seed) * 2 + 1)).cpu().numpy()
    torch.cuda.synchronize()
    return s


def _tau2(case):
    r = np.arange(case["ori"] // 2 + 1)
    return 2e-3 * np.exp(-r / (0.2 * case["ori"]))


def run(state):
    case, e, kind = state["case"], state["e"], state["case"]["kind"]
    if kind == "pool":
        d = state["d"]
        e.reset_sums()
        r = e.expectation_device(d["n"], *_ptrs(d, 0, d["n"]))
        return {"images": r, "sums": e.get_sums()}
    if kind == "fine":
        d = state["d"]
        e.reset_sums()
        r = e.expectation_fine_device(d["n"], *_ptrs(d, 0, d["n"]), state["keys"].data_ptr(), state["cnt"].data_ptr(), state["cap"])
        return {"images": r, "sums": e.get_sums()}
    if kind == "iter":
        # the new model is not installed and the maps are not made references: every pass is the same iteration
        d, n, K = state["d"], case["n"], case["K"]
        e.reset_sums()
        rs = [e.expectation_device(n, *_ptrs(d, p * n, (p + 1) * n)) for p in range(case["pools"])]
        model = e.update_model(install=False)
        vols, power = [], []
        for k in range(K):
            v, tau2, s2, dvp = e.reconstruct(k, _tau2(case), normalise=max(float(model["pdf_class"][k]), 1e-3))
            vols.append(v)
            power.append((s2, dvp))
        return {"images": rs, "model": model, "maps": np.stack(vols), "spectra": np.array(power)}
    if kind == "prep":
        dev = state["dev"]
        out = e.prepare_images(state["images"], state["xoff"], state["yoff"], norm=state["norm"], ctf=state["ctf"], noise=state["noise"],
                               pixel_size=1.5, particle_diameter=1.5 * 0.8 * case["ori"],
                               device_out={k: v.data_ptr() for k, v in dev.items()})
        return {"host": out, "device": dev}
    if kind == "recon":
        v, t, s2, dvp = e.reconstruct(0, state["tau2"], max_iter_preweight=case["iters"], do_map=bool(case["do_map"]))
        return {"map": v, "sigma2": s2, "data_vs_prior": dvp}
    if kind == "fmap":
        ps, corr, _ = e.fourier_map(0, state["vol"], want_grid=False)
        # the installed reference seen through one projection
        re, im = e.project(0, case["cur"], np.eye(3))
        return {"power": ps, "corrected": corr, "slice": (re.astype(np.float32), im.astype(np.float32))}
    if kind == "offl":
        e.reset_sums()
        e.backproject_images(0, state["img"], state["euler"], state["shift"])
        return {"map": e.reconstruct(0, np.zeros(case["ori"] // 2 + 1), do_map=False, minres_map=-1, is_whole_instead_of_half=True)[0]}
    loss = e.proposal_train(case["epochs"], batch=case["batch"], lr=case["lr"])
    return {"loss": loss, "params": e.proposal_get_params()}


# ------------------------------------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    ori, cur = case["ori"], case["cur"]
    dim = case.get("dim", 3)
    F2 = cur * (cur // 2 + 1)
    pad = _pad(cur)
    grid = pad**dim / 2.0
    N = (2 * ori) ** dim
    if kind in ("pool", "fine", "iter", "train"):
        R = 12 * 4 ** case["order"] * 6 * 2 ** case["order"] if dim == 3 else math.ceil(360 / case["psi"])
        T, n = len(rome_amd.translations(case["rng"], 1.0)[0]), case["n"] * case.get("pools", 1)
        cs = case["coarse"] if case["over"] else cur
        coarse = 4.0 * n * case["K"] * R * T * (0.39 * cs * cs)
        w = {"bytes": n * F2 * 12.0 + case["K"] * grid * (8 + 2 * 12), "flops": coarse}
        if kind == "fine":  # 32 fine samples for each given one, and as many rotations projected once
            w = {"bytes": n * F2 * 12.0 + case["K"] * grid * 32, "flops": 1.6 * n * case["median"] * 32 * 8 * 0.39 * cur * cur}
        elif kind == "iter":
            fft = 5.0 * grid * 2 * math.log2(grid * 2)
            w = {"bytes": w["bytes"] + case["K"] * (grid * 12 + ori**dim * 8), "flops": coarse + case["K"] * 10 * fft}
        elif kind == "train":
            H, out = case["hidden"], case["K"] * 4 * 12 * 4 ** case["order"] * 4 + 2
            par = H * (2 * case["coef"] + 2 * H + out)
            steps = case["epochs"] * (case["n"] // case["batch"])
            w = {"bytes": steps * par * 28.0, "flops": 6.0 * par * case["batch"] * steps}
        return w
    if kind == "prep":
        n = case["n"]
        return {"bytes": n * (8.0 * ori * ori * (1 + case["noise"]) + F2 * (16 + 16 + 8 + 8 + 8 + 4)),
                "flops": n * 2 * 2.5 * ori * ori * math.log2(ori * ori)}
    if kind == "fmap":
        return {"bytes": 16.0 * ori**dim + 8 * grid, "flops": 2.5 * N * math.log2(N)}
    fft = 2 * 5.0 * grid * math.log2(2 * grid) * case.get("iters", 10) + 2.5 * N * math.log2(N)
    w = {"bytes": 12.0 * grid + 8.0 * ori**dim, "flops": fft}
    if kind == "offl":
        w = {"bytes": w["bytes"] + case["n"] * F2 * 24.0 + 24.0 * grid, "flops": fft + case["n"] * F2 * 60.0}
    return w


# -------------------------------------------------------------------------------- the calls in 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind in ("pool", "fine", "iter"):
        d = _data(case, seed)
        M = case["K"] * d["D"] * d["PSI"]
        cost = d["n"] * (M * d["T"] if kind != "fine" else 1e5) * (case["coarse"] if case["over"] else case["cur"]) ** 2
        if cost > 3e14 or d["n"] > 1200:
            return None  # more than about 20 seconds in 64 bits
        keys = None
        if kind == "fine":
            k, c, _ = _significance(case, d, seed)
            keys = [torch.sort(k[i, : int(c[i])].long()).values for i in range(d["n"])]
        rs, sums, bp = [], None, None
        for p in range(case.get("pools", 1)):
            r, sums, bp = _estep(case, d, p * case["n"], (p + 1) * case["n"], keys, sums, bp, kind == "iter")
            rs.append(r)
        if kind != "iter":
            return {"images": rs[0], "sums": sums}
        model = _model(case, d, sums)
        vols, spec = [], []
        for k in range(case["K"]):
            v, s2, dvp = _reconstruct(bp[0][k], bp[1][k], case, _tau2(case), 10, True, max(float(model["pdf_class"][k]), 1e-3))
            vols.append(v)
            spec.append((s2, dvp))
        return {"images": rs, "model": model, "maps": np.stack(vols), "spectra": np.array(spec)}
    if kind == "prep":
        return _prep_exact(case, _prep_inputs(case, seed))
    if kind == "fmap":
        vol = _blobs(case["ori"], case["dim"], 100, torch.Generator().manual_seed(int(seed) * 2 + 1))
        G, ps, corr = _fourier_map(vol, case["cur"], True)
        x, y = _half_xy(case["cur"])
        v = _project(G, torch.eye(3, dtype=F64, device=DEV)[None], x, y, (case["cur"] // 2) ** 2)
        return {"power": ps, "corrected": corr, "slice": (v.real, v.imag)}
    if kind in ("recon", "offl"):
        F, ctf, euler, shift = _rotations_grid(None, case, seed)
        ctf = ctf if case.get("ctf", 1) else torch.ones_like(ctf)
        pad, dim = _pad(case["cur"]), case["dim"]
        shape = (pad,) * (dim - 1) + (pad // 2 + 1,)
        data, weight = torch.zeros(shape, dtype=C128, device=DEV), torch.zeros(shape, dtype=F64, device=DEV)
        x, y = _half_xy(case["cur"])
        S = _phase(shift[:, 0], shift[:, 1], x, y, case["ori"])
        _backproject(data, weight, _matrices(euler), F * S * ctf, ctf * ctf, case["cur"])
        if kind == "offl":
            return {"map": _reconstruct(data, weight, case, None, 10, False, 1.0)[0]}
        v, s2, dvp = _reconstruct(data, weight, case, _tau2(case), case["iters"], bool(case["do_map"]), 1.0)
        return {"map": v, "sigma2": s2, "data_vs_prior": dvp}
    return None  # train: steps that round to BF16 by definition have no 64-bit value


def _backproject(data, weight, A, val, wgt, cur, chunk=64):
    x, y = _half_xy(cur)
    px = torch.nonzero((_shell(cur) >= 0) & (x * x + y * y <= (cur // 2) ** 2))[:, 0]
    A = A if data.dim() == 3 else A[:, :2, :2]
    d2, w1 = torch.view_as_real(data).reshape(-1, 2), weight.reshape(-1)
    for q in range(0, len(A), chunk):
        idx, w, neg = _corners(A[q : q + chunk], x[px], y[px], data.shape[-2])
        v, g = val[q : q + chunk][:, px], wgt[q : q + chunk][:, px]
        v = torch.where(neg, v.conj(), v) * (g > 0)
        idx = idx.reshape(-1)
        d2.index_add_(0, idx, torch.view_as_real(v[..., None] * w).reshape(-1, 2))
        w1.index_add_(0, idx, (g[..., None] * w).reshape(-1))


def _weights(d2, prior):
    """diff2 [..] and prior -> (min, weights, sum)."""
    mn = d2.min()
    dd = d2 - mn
    w = torch.where(dd > 700, torch.zeros_like(dd), prior * torch.exp(-dd))
    return mn, w, w.sum()


def _threshold(w, sumw):
    s = torch.sort(w.reshape(-1), descending=True).values
    over = torch.cumsum(s, 0) > 0.999 * sumw
    q = int(torch.nonzero(over)[0, 0]) if bool(over.any()) else s.numel() - 1
    return q + 1, s[q]


def _estep(case, d, a, b, keys, sums, bp, want_bp):
    """The E-step of images a .. b: per-image results, sums and (want_bp) grids, added to those given."""
    ori, cur, K, D, PSI, T, dim = case["ori"], case["cur"], case["K"], d["D"], d["PSI"], d["T"], case["dim"]
    over, R, oriF, n = case["over"], d["D"] * d["PSI"], ori // 2 + 1, b - a
    M, t = K * R, d["tables"]
    up = lambda v: torch.tensor(np.asarray(v), dtype=F64, device=DEV)  # noqa: E731
    x, y = _half_xy(cur)
    sigma2, pdir, prior, tx, ty = up(d["sigma2"]), up(d["pdf_dir"]), up(d["prior"]), up(t["trans_x"]), up(t["trans_y"])
    pdf_m = pdir.reshape(-1).repeat_interleave(PSI)
    k_m = torch.arange(K, device=DEV).repeat_interleave(R)
    if sums is None:
        z = lambda *s: torch.zeros(*s, dtype=F64, device=DEV)  # noqa: E731
        sums = dict(wsum_sigma2_noise=z(case["groups"], oriF), wsum_sumw_group=z(case["groups"]), wsum_pdf_class=z(K),
                    wsum_pdf_direction=z(K, D), wsum_prior_offx=z(K), wsum_prior_offy=z(K), wsum_scalars=z(4))
        if want_bp:
            pad = _pad(cur)
            sh = (K,) + (pad,) * (dim - 1) + (pad // 2 + 1,)
            bp = (torch.zeros(sh, dtype=C128, device=DEV), torch.zeros(sh, dtype=F64, device=DEV))
    NOR, NOT = (8 if dim == 3 else 2, 4) if over else (1, 1)
    euler = lambda p: _matrices(p) if dim == 3 else _matrices(np.stack([0 * p, 0 * p, p], -1))  # noqa: E731
    Ac = euler(t["pose_coarse"].reshape(R, -1) if dim == 3 else t["pose_coarse"])
    pose_f = t["pose_fine"] if over else t["pose_coarse"]
    pose_f = np.asarray(pose_f).reshape(R * NOR, -1)
    Af = euler(pose_f if dim == 3 else pose_f[:, 0])
    sfx, sfy = (up(t["shift_fine_x" if over else "shift_coarse_x"]).reshape(-1), up(t["shift_fine_y" if over else "shift_coarse_y"]).reshape(-1))
    # coarse pixels: the low frequencies of the half-plane
    cs = case["coarse"] if over else cur
    xc, yc = _half_xy(cs)
    mc = _shell(cs)
    pc = torch.nonzero(mc > 0)[:, 0]
    nc = torch.where(yc >= 0, yc, yc + cur)[pc] * (cur // 2 + 1) + xc[pc]
    Sc = _phase(up(t["shift_coarse_x"]), up(t["shift_coarse_y"]), xc[pc], yc[pc], ori)
    if keys is None:
        Fc = torch.cat([_project(d["grids"][k], Ac, xc[pc], yc[pc], (cs // 2) ** 2) for k in range(K)])
        Fc2 = torch.cat([Fc.real, Fc.imag], 1)
        Fa = Fc.abs() ** 2
    mf = _shell(cur)
    pf = torch.nonzero(mf >= 0)[:, 0]
    xf, yf, mf = x[pf], y[pf], mf[pf]
    Sf = _phase(sfx, sfy, xf, yf, ori)
    nan = float("nan")
    out = dict(meta=torch.zeros(n, 9, dtype=F64), nr_sign=torch.zeros(n, dtype=torch.int32), argmax=torch.zeros(n, 6, dtype=torch.int32))
    for q in ("min_diff2", "sum_weight", "sig_weight", "min_diff2_coarse", "sum_weight_coarse", "sig_weight_coarse", "wsum_norm_correction"):
        out[q] = torch.full((n,), nan, dtype=F64)
    for i in range(n):
        g = int(d["group"][a + i])
        X, ctf, hx = d["F"][a + i].to(C128), d["ctf"][a + i].double(), d["hx"][a + i]
        ox, oy = d["offx"][a + i], d["offy"][a + i]
        s2o = d["sigma2_offset"]
        td = (tx[None] + ox - prior[0][:, None]) ** 2 + (ty[None] + oy - prior[1][:, None]) ** 2
        pdf_off = torch.exp(td / (-2 * s2o)) / (2 * PI * s2o)  # [K][T]
        if keys is None:
            minv = 1 / sigma2[g][mc[pc]]
            XS = X[nc][None] * Sc
            C = Fc2 @ torch.cat([(XS.real * minv * ctf[nc]), (XS.imag * minv * ctf[nc])], 1).T
            d2 = 0.5 * ((Fa @ (minv * ctf[nc] ** 2))[:, None] - 2 * C + (minv * X[nc].abs() ** 2).sum() + hx)
            mn, w, sw = _weights(d2, pdf_m[:, None] * pdf_off[k_m])
            cnt, thr = _threshold(w, sw)
            out["nr_sign"][i], out["min_diff2_coarse"][i], out["sum_weight_coarse"][i], out["sig_weight_coarse"][i] = cnt, mn, sw, thr
            sel = torch.nonzero((w >= thr).reshape(-1))[:, 0]
        else:
            sel = keys[i]
            out["nr_sign"][i] = len(sel)
        minv = torch.where(mf > 0, 1 / sigma2[g][mf], torch.zeros_like(sigma2[g][mf]))
        Xf, cf = X[pf], ctf[pf]
        if over:
            mu, mi = torch.unique(sel // T, return_inverse=True)
            tu, ti = torch.unique(sel % T, return_inverse=True)
        else:
            mu, tu = torch.arange(M, device=DEV), torch.arange(T, device=DEV)
        rot = (mu % R)[:, None] * NOR + torch.arange(NOR, device=DEV)[None]
        P = torch.zeros(len(mu), NOR, len(pf), dtype=C128, device=DEV)
        for k in torch.unique(mu // R).tolist():
            s = mu // R == k
            P[s] = _project(d["grids"][k], Af[rot[s].reshape(-1)], xf, yf, (cur // 2) ** 2).reshape(-1, NOR, len(pf))
        P = (P * cf).reshape(-1, len(pf))
        St = Sf.reshape(T, NOT, -1)[tu].reshape(-1, len(pf))
        XS = Xf[None] * St
        if over:
            cross = torch.cat([P.real * minv, P.imag * minv], 1) @ torch.cat([XS.real, XS.imag], 1).T
            d2 = 0.5 * (((P.abs() ** 2) @ minv)[:, None] - 2 * cross + (minv * Xf.abs() ** 2).sum() + hx)
            d2 = d2.reshape(len(mu), NOR, len(tu), NOT).permute(0, 2, 1, 3)  # [m][t][o][ot]
            ok = torch.zeros(len(mu), len(tu), dtype=torch.bool, device=DEV)
            ok[mi, ti] = True
            d2 = torch.where(ok[:, :, None, None], d2, torch.full_like(d2, float("inf")))
            pr = pdf_m[mu][:, None] * pdf_off[mu // R][:, tu]
            mn, w, sw = _weights(d2, pr[:, :, None, None])
        else:
            w, d2 = w[:, :, None, None], d2[:, :, None, None]
        flat = w.reshape(-1)
        best = int(torch.nonzero(flat == flat.max())[0, 0])
        _, thr = _threshold(flat[flat > 0], sw)
        out["min_diff2"][i], out["sum_weight"][i], out["sig_weight"][i] = mn, sw, thr
        q = np.unravel_index(best, tuple(w.shape))
        m, tb = int(mu[q[0]]), int(tu[q[1]])
        out["argmax"][i] = torch.tensor([m // R, (m % R) // PSI, m % PSI, q[2], tb, q[3]])
        p = pose_f[(m % R) * NOR + q[2]]
        wrap = lambda v: v - 360 if v > 180 else v + 360 if v < -180 else v  # noqa: E731
        ang = [p[0], p[1], p[2]] if dim == 3 else [0, 0, wrap(p[0])]
        # sums over the significant samples: W [rotations][shifts]
        W = torch.where(w >= thr, w / sw, torch.zeros_like(w)).permute(0, 2, 1, 3).reshape(len(mu) * NOR, len(tu) * NOT)
        live = torch.nonzero(W.sum(1) > 0)[:, 0]
        W, P, mk = W[live], P[live], mu.repeat_interleave(NOR)[live]
        if case["dim"] == 3 and not over:
            W = W * 0
        wr, wt = W.sum(1), W.sum(0)
        e2 = wr @ (P.abs() ** 2) + wt @ (XS.abs() ** 2) - 2 * ((W.T.to(C128) @ P) * XS.conj()).real.sum(0)
        sums["wsum_sigma2_noise"][g].index_add_(0, mf, e2)
        wn = e2.sum()
        sums["wsum_sumw_group"][g] += wr.sum()
        sums["wsum_pdf_class"].index_add_(0, mk // R, wr)
        sums["wsum_pdf_direction"].view(-1).index_add_(0, mk // PSI, wr)
        sx, sy = (v.reshape(T, NOT)[tu].reshape(-1) for v in (sfx, sfy))
        far = (prior[0][mk // R][:, None] - ox - sx) ** 2 + (prior[1][mk // R][:, None] - oy - sy) ** 2
        sums["wsum_scalars"][0] += (W * far).sum()
        if dim == 2:
            sums["wsum_prior_offx"].index_add_(0, mk // R, W @ (ox + sx))
            sums["wsum_prior_offy"].index_add_(0, mk // R, W @ (oy + sy))
        if want_bp:
            mb = torch.where(mf == 0, 1 / sigma2[g][0], minv) * cf
            val = torch.zeros(len(live), len(x), dtype=C128, device=DEV)
            wgt = torch.zeros(len(live), len(x), dtype=F64, device=DEV)
            val[:, pf] = W.to(C128) @ (St * (Xf * mb))
            wgt[:, pf] = wr[:, None] * (mb * cf)
            ro = rot.reshape(-1)[live]
            for k in torch.unique(mk // R).tolist():
                s = mk // R == k
                _backproject(bp[0][k], bp[1][k], Af[ro[s]], val[s], wgt[s], cur)
        hi = d["power"][a + i][cur // 2 + 1 :]
        sums["wsum_sigma2_noise"][g][cur // 2 + 1 :] += hi
        wn = wn + hi.sum()
        norm = d["norm"][a + i] * torch.sqrt(2 * wn)
        dll = torch.log(sw) - mn - torch.log(2 * PI * sigma2[g][mf[mf > 0]]).sum()
        pmax = flat[best] / sw
        out["wsum_norm_correction"][i] = wn
        out["meta"][i] = torch.tensor([float(v) for v in (pmax, m // R + 1, *ang, ox + sfx[tb * NOT + q[3]], oy + sfy[tb * NOT + q[3]], norm, dll)], dtype=F64)
        sums["wsum_scalars"][1] += dll
        sums["wsum_scalars"][2] += pmax
        sums["wsum_scalars"][3] += norm
    return out, sums, bp


def _model(case, d, s):
    sh = _shell(case["ori"])
    npix = torch.bincount(sh[sh >= 0], minlength=case["ori"] // 2 + 1).to(F64)
    wk, sc = s["wsum_pdf_class"], s["wsum_scalars"]
    sw = wk.sum()
    p = [s["wsum_prior_offx"], s["wsum_prior_offy"]]
    p = [torch.where(wk > 0, v / wk, torch.zeros_like(wk)) if case["dim"] == 2 else torch.zeros_like(wk) for v in p]
    return dict(sigma2_noise=s["wsum_sigma2_noise"] / (2 * s["wsum_sumw_group"][:, None] * npix[None]), pdf_class=wk / sw,
                pdf_direction=s["wsum_pdf_direction"] / sw, prior_offx=p[0], prior_offy=p[1],
                scalars=torch.stack([sc[0] / (2 * sw), sc[3] / sw, sc[1], sc[2] / sw]))


def _blob_table():
    w = np.arange(10000) * (0.5 / 10000)
    v = 2 * PI * 3.8 * w
    sig = np.sqrt(np.abs(225.0 - v * v))
    with np.errstate(over="ignore", invalid="ignore"):
        out = np.where(v > 15.0, np.sin(sig) / sig - np.cos(sig), np.cosh(np.minimum(sig, 16)) - np.sinh(np.minimum(sig, 16)) / sig)
    out = out / sig**2
    return torch.tensor(out / out[0], device=DEV)


def _reconstruct(data, weight, case, tau2, iters, do_map, normalise):
    ori, cur, dim = case["ori"], case["cur"], case["dim"]
    r_max, P, N, oriF = cur // 2, _pad(cur), 2 * ori, ori // 2 + 1
    PF, c, m2 = P // 2 + 1, P // 2, 4 * (cur // 2) ** 2
    osc = 8.0 if dim == 3 else 4.0
    axes = tuple(range(dim))
    data, weight = data.clone(), weight.clone()
    p0, w0 = data[..., 0].clone(), weight[..., 0].clone()
    fl = torch.flip(p0, tuple(range(dim - 1)))
    data[..., 0], weight[..., 0] = p0 + fl.conj(), w0 + torch.flip(w0, tuple(range(dim - 1)))
    mid = (c,) * (dim - 1)  # the origin is its own mirror image and stays as it is
    data[mid + (0,)], weight[mid + (0,)] = p0[mid], w0[mid]
    order = _signed(P, PF) + c  # centred -> FFT order
    for ax in range(dim - 1):
        data, weight = data.index_select(ax, order), weight.index_select(ax, order)
    k = _signed(P, PF)
    r2 = _rad2(*([k] * (dim - 1)), torch.arange(PF, device=DEV))
    zero = torch.zeros((), dtype=F64, device=DEV)
    Fw = torch.where(r2 <= m2, weight, zero)
    ins = r2 < m2
    sh = torch.floor(torch.sqrt(r2[ins].to(F64)) / 2 + 0.5).long()
    add = lambda v: _shell_sums(sh, v, ori)  # noqa: E731
    ct, s0 = add(torch.ones_like(sh, dtype=F64)), add(osc * Fw[ins])
    sigma2 = torch.where(s0 > 1e-10, ct / s0.clamp(min=1e-300), torch.zeros_like(s0))
    dvp = torch.zeros(oriF, dtype=F64, device=DEV)
    if do_map:
        tt = torch.tensor(tau2, device=DEV)[sh]
        inv = Fw[ins]
        it = torch.where(tt > 0, 1 / (osc * tt.clamp(min=1e-300)), 1 / (0.001 * inv))
        v = add(inv / it)
        dvp = torch.where(torch.arange(oriF, device=DEV) > r_max, zero, torch.where(ct < 0.001, zero + 999, v / ct.clamp(min=1)))
        Fw[ins] = torch.where(sh >= 5, inv + it, inv)
    Fw, data = Fw / normalise, data / normalise
    nw = ins.to(F64)
    tab = _blob_table()
    s = _signed(P, P // 2)
    idx = (torch.sqrt(_rad2(*([s] * dim)).to(F64)) / (2 * ori) / (0.5 / 10000)).long()
    blob = torch.where(idx < 10000, tab[idx.clamp(max=9999)], zero)
    for _ in range(iters):
        Mr = torch.fft.irfftn((nw * Fw).to(C128), s=(P,) * dim, dim=axes) * blob
        w = torch.fft.rfftn(Mr, dim=axes).abs().clamp(min=1e-6)
        nw = torch.where(ins, nw / w, nw)
    F = torch.where(r2 <= m2, data, torch.zeros_like(data)) * nw
    NF = N // 2 + 1
    kn = torch.arange(P, device=DEV) - P // 2
    if NF < PF:
        kn = kn[(kn >= NF - N) & (kn < NF)]
    nj = min(NF, PF)
    src, dst = kn % P, kn % N
    F = torch.where(r2 <= (PF - 1) ** 2, F, torch.zeros_like(F)) if NF >= PF else F
    big = torch.zeros((N,) * (dim - 1) + (NF,), dtype=C128, device=DEV)
    if dim == 3:
        big[dst[:, None], dst[None, :], :nj] = F[src[:, None], src[None, :], :nj]
        scale = N**3 / (8.0 * ori)
    else:
        big[dst, :nj] = F[src, :nj]
        scale = N**2 / 4.0
    vol = torch.roll(torch.fft.irfftn(big, s=(N,) * dim, dim=axes), (N // 2,) * dim, axes) * scale
    o = N // 2 - ori // 2
    vol = vol[(slice(o, o + ori),) * dim]
    r = _radius(ori, dim)
    rad = ori / 2.0
    rc = torch.where(r > rad + 3, zero + 1, torch.where(r >= rad, 0.5 + 0.5 * torch.cos(PI * (rad + 3 - r) / 3), zero))
    bg = (rc * vol).sum() / rc.sum()
    vol = ((1 - rc) * vol + rc * bg) / _sinc2(ori, dim)
    return vol.cpu().numpy(), sigma2.cpu().numpy(), dvp.cpu().numpy()


def _prep_exact(case, s):
    ori, cur, n = case["ori"], case["cur"], case["n"]
    img = torch.tensor(s["images"], device=DEV)
    if case["norm"]:
        img = img * 1.1 / torch.tensor(s["norm"], device=DEV)[:, None, None]
    rnd = lambda v: np.where(v >= 0, np.floor(v + 0.5), -np.floor(-v + 0.5))  # noqa: E731
    ox, oy = rnd(s["xoff"]), rnd(s["yoff"])
    mv = torch.zeros_like(img)
    ax = torch.arange(ori, device=DEV)
    sy = ax[None] - torch.tensor(oy, device=DEV).long()[:, None]
    sx = ax[None] - torch.tensor(ox, device=DEV).long()[:, None]
    ok = ((sy >= 0) & (sy < ori))[:, :, None] & ((sx >= 0) & (sx < ori))[:, None, :]
    i = torch.arange(n, device=DEV)[:, None, None]
    mv = torch.where(ok, img[i, sy.clamp(0, ori - 1)[:, :, None], sx.clamp(0, ori - 1)[:, None, :]], mv)
    r = _radius(ori, 2)
    rad, width = 0.4 * ori, 5.0
    one = torch.ones_like(r)
    rc = torch.where(r > rad + width, one, torch.where(r >= rad, 0.5 + 0.5 * torch.cos(PI * (rad + width - r) / width), 0 * one))
    fill = torch.tensor(s["noise"], device=DEV) if case["noise"] else ((mv * rc).sum((1, 2)) / rc.sum())[:, None, None]
    masked = (1 - rc) * mv + rc * fill
    ft = lambda v: torch.fft.rfft2(torch.roll(v, (ori // 2, ori // 2), (1, 2))) / ori**2  # noqa: E731
    Fn, Fm = ft(mv), ft(masked)
    rows = _signed(cur, cur // 2 + 1) % ori
    win = lambda v: v[:, rows, : cur // 2 + 1].reshape(n, -1)  # noqa: E731
    oF = ori // 2 + 1
    power = torch.zeros(n, oF, dtype=F64, device=DEV)
    if cur < ori:
        sh = _shell(ori)
        px = torch.nonzero(sh > 0)[:, 0]
        power.index_add_(1, sh[px], (Fm.reshape(n, -1)[:, px].abs()) ** 2)
    hx = power[:, cur // 2 + 1 :].sum(1)
    ctf = _ctf(cur, ori, 1.5, torch.tensor(s["ctf"], device=DEV)) if case["ctf"] else torch.ones(n, cur * (cur // 2 + 1), dtype=F64, device=DEV)
    wn, wm = win(Fn), win(Fm)
    host = dict(fmask_re=wm.real, fmask_im=wm.imag, fnomask_re=wn.real, fnomask_im=wn.imag, fctf=ctf, highres_Xi2=hx, power_img=power,
                old_offx=ox, old_offy=oy)
    dev = dict(fmask=torch.view_as_real(wm), fnomask=torch.view_as_real(wn), fctf=ctf, highres_Xi2=hx, power_img=power, old_offx=ox, old_offy=oy)
    return {"host": host, "device": dev}
