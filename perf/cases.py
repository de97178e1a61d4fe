"""Measured cases: the calls a reconstruction program makes through omega_amd's public entry points.

Emission (PET) data are rings of detectors sampled as parallel-chord sinograms, in 2-D (direct planes,
one per image slice) or 3-D (span-1 ring pairs); transmission (CT) data are a circular cone-beam
trajectory with a flat panel. Phantoms are random ellipsoids in a uniform cylinder; measurements are
Poisson counts of their analytic line integrals (CT: the integrals with Gaussian noise), so inputs do
not depend on the projectors under measurement.

Kinds: ``osem`` (whole OSEM / OSL-OSEM iterations, sensitivity images included, with one of the
projectors), ``project`` (one forward or back projection of a 3-D PET subset), ``frames`` (one subset
step of every frame of a dynamic study), ``ct`` (one distance-driven forward or back projection of a
view subset) and ``unet`` (forward and backward pass of the warm-start network).
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from omega_amd.dynamic import FramesOSEM
from omega_amd.projector import projectorClass
from omega_amd.recon import OSEMRunner
from omega_amd.unet import UNet3D

DEV = "cuda"
EPPS = 1e-5
LIGHT = 2.99792458e11      # mm / s


def _pet2d(name, projector, nx, ny, nz, ndist, nang, subsets, iters, beta=0.0, randoms=False, tof=0, atten=False):
    return {"name": name, "kind": "osem", "projector": projector, "nx": nx, "ny": ny, "nz": nz, "fov": 320.0,
            "axial": 2.5 * nz, "rings": 0, "mrd": 0, "radius": 400.0, "ndist": ndist, "nang": nang,
            "pitch": 320.0 / ndist, "subsets": subsets, "subset_type": 8, "iters": iters, "beta": beta,
            "randoms": randoms, "tof": tof, "atten": atten, "counts": 4.0 * nz * ndist * nang}


def _pet3d(name, kind, rings, ring_pitch, ndist, nang, radius, fov, nx, ny, nz, subsets, subset_type=8, mrd=None, **kw):
    c = {"name": name, "kind": kind, "projector": 1, "nx": nx, "ny": ny, "nz": nz, "fov": fov,
         "axial": rings * ring_pitch, "rings": rings, "mrd": rings - 1 if mrd is None else mrd, "radius": radius,
         "ndist": ndist, "nang": nang, "pitch": math.pi * radius / (2 * ndist), "subsets": subsets,
         "subset_type": subset_type, "iters": 1, "beta": 0.0, "randoms": False, "tof": 0, "atten": False,
         "counts": 2e7}
    c.update(kw)
    return c


def _ct(name, op, n, voxel, views, subsets, rows, cols, pixel):
    return {"name": name, "kind": "ct", "op": op, "nx": n[0], "ny": n[1], "nz": n[2], "voxel": voxel, "views": views,
            "subsets": subsets, "rows": rows, "cols": cols, "pixel": pixel, "sod": 700.0, "sdd": 1000.0}


def listed():
    return [
        # a small animal scanner's iteration with the relative difference prior (angle subsets): every launch is
        # tiny, so latency and the number of launches count
        _pet3d("osl_pet3d_small", "osem", 8, 4.0, 48, 48, 150.0, 160.0, 40, 40, 15, 4, 4, beta=0.01, counts=5e5),
        # the 2-D plane PET reconstruction most users run: one iteration that also makes the sensitivity
        # images and one that reads them
        _pet2d("osem_pet2d", 1, 128, 128, 63, 128, 160, 8, 2),
        # odd sizes, a non-square image, prior and randoms term
        _pet2d("osl_pet2d_odd", 1, 109, 97, 41, 142, 91, 5, 2, beta=0.01, randoms=True),
        # time of flight with attenuation
        _pet2d("osem_pet2d_tof", 1, 128, 128, 63, 128, 160, 8, 1, tof=17, atten=True),
        # the other two emission projectors on the same scanner
        _pet2d("osem_pet2d_orth", 2, 128, 128, 63, 128, 160, 8, 2),
        _pet2d("osem_pet2d_interp", 4, 128, 128, 63, 128, 160, 8, 2),
        # a clinical 3-D scanner: one of 16 subsets, each direction as custom algorithms call it
        _pet3d("pet3d_forward", "project", 32, 4.0, 224, 224, 400.0, 320.0, 128, 128, 63, 16, op="forward"),
        _pet3d("pet3d_backward", "project", 32, 4.0, 224, 224, 400.0, 320.0, 128, 128, 63, 16, op="backward"),
        # a dynamic study: one subset step of all frames
        _pet3d("frames_pet3d", "frames", 32, 4.0, 224, 224, 400.0, 320.0, 128, 128, 63, 16, frames=8, counts=4e6),
        # cone-beam CT: one of 8 view subsets of 360 views, each direction
        _ct("ct_forward", "forward", (256, 256, 256), 0.5, 360, 8, 512, 384, 0.8),
        _ct("ct_backward", "backward", (256, 256, 256), 0.5, 360, 8, 512, 384, 0.8),
        # training the warm start: the network's forward pass, loss and all parameter gradients
        {"name": "unet_gradients", "kind": "unet", "nx": 128, "ny": 128, "nz": 63},
    ]


def _spread(rng, lo, hi):
    """Whole number in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["small", "osem2d", "osl2d", "tof", "orth", "interp", "forward", "backward", "frames", "ctf",
                       "ctb", "unet"])
    if kind == "small":
        rings, subsets = rng.randint(4, 12), rng.choice([2, 4, 6])
        n = rng.randint(6, 20)
        return {k: v for k, v in _pet3d("", "osem", rings, 4.0, rng.randrange(32, 80, 2), subsets * n, 150.0, 160.0,
                                        *(2 * [rng.randint(24, 64)]), 2 * rings - 1, subsets, 4, beta=0.01,
                                        counts=5e5).items() if k != "name"}
    if kind in ("osem2d", "osl2d", "tof", "orth", "interp"):
        nx = rng.randint(96 if kind == "orth" else 48, 132)     # the 2.5 mm tube needs voxels of about its width
        ny = nx
        if rng.random() < 0.5:
            nx = ny = 4 * (nx // 4)
        elif rng.random() < 0.5:
            ny = rng.randint(96 if kind == "orth" else 48, 132)
        nang = rng.randint(50, 160)
        if nx != ny:
            nang |= 1
        projector = {"orth": 2, "interp": 4}.get(kind, 1)
        subsets = rng.randint(3, 10)
        osl = kind == "osl2d" or (projector == 4 and rng.random() < 0.5)
        c = _pet2d("", projector, nx, ny, _spread(rng, 10, 63), 2 * rng.randint(32, 72), nang, subsets,
                   1 if kind == "tof" else 2, beta=0.01 if osl else 0.0, randoms=rng.random() < 0.5,
                   tof=rng.choice([5, 9, 13, 17]) if kind == "tof" else 0,
                   atten=kind == "tof" or (projector != 4 and rng.random() < 0.3))
        return {k: v for k, v in c.items() if k != "name"}
    if kind in ("forward", "backward", "frames"):
        rings = _spread(rng, 10, 32)
        nx = rng.randint(64, 144)
        ny = nx if rng.random() < 0.6 else rng.randint(64, 144)
        ndist, nang = 2 * rng.randint(50, 112), rng.randint(80, 224)
        if nx != ny:
            nang |= 1
        mrd = rng.randint(rings // 2, rings - 1)
        planes = rings + sum(2 * (rings - d) for d in range(1, mrd + 1))
        lors = planes * ndist * nang
        subsets = max(rng.randint(4, 20), math.ceil(lors / 3.0e6))
        kw = {"op": kind} if kind != "frames" else {"frames": rng.choice([2, 4, 6, 8])}
        return {k: v for k, v in _pet3d("", "frames" if kind == "frames" else "project", rings, 4.0, ndist, nang, 400.0,
                                        320.0, nx, ny, rng.choice([2 * rings - 1, rings | 1]), subsets, 8, mrd,
                                        counts=4e6, **kw).items() if k != "name"}
    if kind in ("ctf", "ctb"):
        n = (rng.randint(80, 256), rng.randint(80, 256), rng.randint(64, 256))
        rows, cols = rng.randint(160, 512), rng.randint(120, 384)
        voxel = 128.0 / max(n)
        pixel = 0.8 * 512.0 / max(rows, cols)
        views = rng.randint(90, 360)
        c = _ct("", "forward" if kind == "ctf" else "backward", n, voxel, views, max(8, views // 45 + 1), rows, cols,
                pixel)
        return {k: v for k, v in c.items() if k != "name"}
    return {"kind": "unet", "nx": 4 * rng.randint(12, 32), "ny": 4 * rng.randint(12, 32), "nz": _spread(rng, 12, 63)}


# ---- geometry tables -------------------------------------------------------------------------------------
def _ring_xy(c):
    """[xs, ys, xd, yd] per (radial bin, angle), radial fastest: chords of the detector ring."""
    s = (np.arange(c["ndist"]) - (c["ndist"] - 1) / 2.0) * c["pitch"]
    phi = np.arange(c["nang"]) * math.pi / c["nang"]
    S, P = np.meshgrid(s, phi, indexing="xy")
    h = np.sqrt(np.maximum(c["radius"] ** 2 - S * S, 0.0))
    co, si = np.cos(P), np.sin(P)
    return np.stack([S * co + h * si, S * si - h * co, S * co - h * si, S * si + h * co], -1).reshape(-1, 4).astype(np.float32)


def _planes(c):
    """[zs, zd] per plane: direct planes at the slice centres, or ring pairs by ring difference."""
    if not c["rings"]:
        z = (np.arange(c["nz"]) + 0.5) * (c["axial"] / c["nz"]) - c["axial"] / 2
        return np.stack([z, z], -1).astype(np.float32)
    pos = (np.arange(c["rings"]) + 0.5) * (c["axial"] / c["rings"]) - c["axial"] / 2
    out = []
    for d in range(c["mrd"] + 1):
        for r in range(c["rings"] - d):
            out.append((pos[r], pos[r + d]))
        if d:
            for r in range(c["rings"] - d):
                out.append((pos[r + d], pos[r]))
    return np.asarray(out, np.float32)


def _ct_tables(c):
    a = np.arange(c["views"]) * 2 * math.pi / c["views"]
    co, si, o = np.cos(a), np.sin(a), np.zeros_like(a)
    R, D = c["sod"], c["sdd"]
    x = np.stack([R * co, R * si, o, -(D - R) * co, -(D - R) * si, o], -1).astype(np.float32)
    uv = np.stack([-si * c["pixel"], co * c["pixel"]], -1).astype(np.float32)
    return x, uv


def _ct_subset(c):
    return np.arange(1, c["views"], c["subsets"])     # subset 1 of type 8


def _tof_tables(c):
    """Standard deviation and bin centres (mm): 400 ps FWHM, 140 ps bins, central bin first."""
    sigma = np.float32(LIGHT * 400e-12 / 2 / (2 * math.sqrt(2 * math.log(2))))
    h = c["tof"] // 2
    order = [0] + [s * k for k in range(1, h + 1) for s in (1, -1)]
    return sigma, (np.asarray(order, np.float64) * -140e-12 * LIGHT / 2).astype(np.float32)


# ---- phantoms and data ------------------------------------------------------------------------------------
def _ellipsoids(seed, fov, axial, n=8, lo=0.5, hi=2.0):
    rng = random.Random(seed)
    out = []
    for _ in range(n):
        r, t = 0.3 * fov * math.sqrt(rng.random()), rng.uniform(0, 2 * math.pi)
        out.append((r * math.cos(t), r * math.sin(t), rng.uniform(-0.3, 0.3) * axial, rng.uniform(0.04, 0.16) * fov,
                    rng.uniform(0.04, 0.16) * fov, rng.uniform(0.1, 0.4) * axial, rng.uniform(lo, hi)))
    return out


def _image(ells, base, n, size):
    """Voxel image, x fastest: cylinder of value ``base`` plus the ellipsoids."""
    ax = [(torch.arange(k, dtype=torch.float32, device=DEV) + 0.5) * (s / k) - s / 2 for k, s in zip(n, size)]
    x, y, z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    img = torch.where((x / (0.45 * size[0])) ** 2 + (y / (0.45 * size[1])) ** 2 < 1, base, 0.0).expand(n[2], n[1], n[0]).clone()
    for cx, cy, cz, ex, ey, ez, act in ells:
        img += act * (((x - cx) / ex) ** 2 + ((y - cy) / ey) ** 2 + ((z - cz) / ez) ** 2 < 1)
    return img.reshape(-1).contiguous()


def _chords(s, v, ell):
    """Lengths inside one ellipsoid of the lines s + t v (broadcast tensors of 3 components each)."""
    A = B = C = 0.0
    for k in range(3):
        q, w = (s[k] - ell[k]) / ell[3 + k], v[k] / ell[3 + k]
        A, B, C = A + w * w, B + q * w, C + q * q
    disc = (B * B - A * (C - 1.0)).clamp_min(0.0)
    return 2.0 * disc.sqrt() / A * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2).sqrt()


def _pet_means(c, ells, base, acts=None):
    """Line integrals [frames, planes, bins] of the phantom, per plane chunk (a generator)."""
    xy = torch.as_tensor(_ring_xy(c), device=DEV)
    z = torch.as_tensor(_planes(c), device=DEV)
    cyl = (0.0, 0.0, 0.0, 0.45 * c["fov"], 0.45 * c["fov"], 50.0 * c["axial"], base)
    for p0 in range(0, z.shape[0], 64):
        zz = z[p0:p0 + 64]
        s = (xy[None, :, 0], xy[None, :, 1], zz[:, :1])
        v = (xy[None, :, 2] - s[0], xy[None, :, 3] - s[1], zz[:, 1:] - zz[:, :1])
        F = 1 if acts is None else len(acts)
        out = torch.zeros((F, zz.shape[0], xy.shape[0]), device=DEV)
        out += base * _chords(s, v, cyl)
        for e, ell in enumerate(ells):
            ch = _chords(s, v, ell)
            for f in range(F):
                out[f] += (ell[6] if acts is None else float(acts[f][e])) * ch
        yield p0, out


def _subset_planes(c, n_planes):
    return [list(range(k, n_planes, c["subsets"])) for k in range(c["subsets"])]


def _pet_counts(c, seed, acts=None):
    """Poisson counts [frames, planes, bins] in sinogram order (with TOF: planes, bins x TOF bins apart)."""
    ells = _ellipsoids(seed, c["fov"], c["axial"])
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 1)
    mean = torch.cat([m for _, m in _pet_means(c, ells, 0.1, acts)], 1)
    mean *= c["counts"] / mean[0].sum(dtype=torch.float64).item()
    if c["tof"]:
        sigma, cen = _tof_tables(c)
        w = np.exp(-0.5 * cen.astype(np.float64) ** 2 / (float(sigma) ** 2 + 70.0 ** 2))
        mean = mean * torch.as_tensor(w / w.sum(), dtype=torch.float32, device=DEV)[:, None, None]
    y = torch.empty_like(mean)
    for f in range(mean.shape[0]):
        y[f] = torch.poisson(mean[f], generator=g)
    return y, mean


def _subset_order(c, y):
    """[frames, planes, bins] -> per subset [frames, LORs of the subset] (subset types 8 and 4)."""
    if c["subset_type"] == 8:
        return [y[:, p].reshape(y.shape[0], -1) for p in _subset_planes(c, y.shape[1])]
    q = y.reshape(y.shape[0], y.shape[1], c["nang"], c["ndist"])
    return [q[:, :, k::c["subsets"]].reshape(y.shape[0], -1) for k in range(c["subsets"])]


def _mu_image(c):
    x = (np.arange(c["nx"]) + 0.5) * (c["fov"] / c["nx"]) - c["fov"] / 2
    y = (np.arange(c["ny"]) + 0.5) * (c["fov"] / c["ny"]) - c["fov"] / 2
    m = np.where(x[None, :] ** 2 + y[:, None] ** 2 < 120.0 ** 2, 0.0096, 0.0).astype(np.float32)
    return np.ascontiguousarray(np.broadcast_to(m, (c["nz"],) + m.shape)).reshape(-1)


def _projector(c):
    p = projectorClass()
    p.Nx, p.Ny, p.Nz = c["nx"], c["ny"], c["nz"]
    if c["kind"] == "ct":
        p.CT, p.projector_type = True, 5
        p.FOVa_x, p.FOVa_y, p.axial_fov = c["nx"] * c["voxel"], c["ny"] * c["voxel"], c["nz"] * c["voxel"]
        x, uv = _ct_tables(c)
        p.x, p.z = x.reshape(-1), uv.reshape(-1)
        p.nRowsD, p.nColsD = c["rows"], c["cols"]
        p.dPitchX = p.dPitchY = c["pixel"]
    else:
        p.FOVa_x, p.FOVa_y, p.axial_fov = c["fov"], c["fov"], c["axial"]
        p.projector_type = c["projector"]
        p.x, p.z = _ring_xy(c).reshape(-1), _planes(c).reshape(-1)
        p.Ndist, p.Nang = c["ndist"], c["nang"]
        if c["projector"] == 2:
            p.tube_width_xy = p.tube_width_z = 2.5
        if c["tof"]:
            p.TOF_bins = p.TOF_bins_used = c["tof"]
            sigma, p.TOFCenter = _tof_tables(c)
            p.sigma_x = float(sigma)
        if c["atten"]:
            p.attenuation_correction = True
            p.vaimennus = _mu_image(c)
    p.subsets = c["subsets"]
    p.subsetType = c.get("subset_type", 8)
    p.addProjector()
    p.initProj()
    return p


# ---- the network's inputs ----------------------------------------------------------------------------------
LAYERS = [("e1a", 16, 16), ("e1b", 16, 16), ("e2a", 16, 32), ("e2b", 32, 32), ("bta", 32, 64), ("btb", 64, 64),
          ("d2a", 96, 32), ("d2b", 32, 32), ("d1a", 48, 16), ("d1b", 16, 16)]


def _unet_params(seed):
    rng = np.random.default_rng(seed)
    out = {}
    for name, cin, cout in LAYERS:
        fan = 27 * (1 if name == "e1a" else cin)
        out[name + ".w"] = rng.normal(0.0, math.sqrt(2.0 / fan), (27, cout, cin)).astype(np.float32)
        out[name + ".b"] = rng.normal(0.0, 0.05, cout).astype(np.float32)
    out["head.w"] = rng.normal(0.0, 0.1, 16).astype(np.float32)
    out["head.b"] = np.zeros(1, np.float32)
    return out


def _unet_images(c, seed):
    n, size = (c["nx"], c["ny"], c["nz"]), (2.5 * c["nx"], 2.5 * c["ny"], 2.5 * c["nz"])
    target = _image(_ellipsoids(seed, min(size[:2]), size[2]), 0.1, n, size)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 2)
    image = (target * (1.0 + 0.3 * torch.randn(target.shape, device=DEV, generator=g))).clamp_min(0.0)
    return image, target


# ---- prepare / run -----------------------------------------------------------------------------------------
def prepare(case, seed):
    c = case
    if c["kind"] == "unet":
        net = UNet3D(c["nx"], c["ny"], c["nz"], params=_unet_params(seed), device=DEV)
        image, target = _unet_images(c, seed)
        return {"c": c, "net": net, "image": image, "target": target, "mask": net.mask()}
    p = _projector(c)
    if c["kind"] == "ct":
        ells = _ct_ellipsoids(c, seed)
        size = tuple(k * c["voxel"] for k in (c["nx"], c["ny"], c["nz"]))
        if c["op"] == "forward":
            return {"c": c, "p": p, "x": _image(ells, 0.004, (c["nx"], c["ny"], c["nz"]), size)}
        return {"c": c, "p": p, "y": _ct_data(c, seed)}
    if c["kind"] == "project":
        n, size = (c["nx"], c["ny"], c["nz"]), (c["fov"], c["fov"], c["axial"])
        if c["op"] == "forward":
            return {"c": c, "p": p, "x": _image(_ellipsoids(seed, c["fov"], c["axial"]), 0.1, n, size)}
        return {"c": c, "p": p, "y": _ratio_data(c, seed)}
    if c["kind"] == "frames":
        y, _ = _pet_counts(c, seed, _frame_activities(c, seed))
        meas = torch.cat(_subset_order(c, y), 1)
        del y
        run_ = FramesOSEM(p, meas)
        run_.sensitivity()
        return {"c": c, "p": p, "run": run_}
    y, mean = _pet_counts(c, seed)
    parts = _subset_order(c, y)
    add = None
    if c["randoms"]:
        add = torch.cat([m.reshape(-1) for m in _subset_order(c, 0.2 * mean[:1] + 0.05 * mean.mean())])
    return {"c": c, "p": p, "run": OSEMRunner(p, torch.cat([q.reshape(-1) for q in parts]), epps=EPPS, beta=c["beta"],
                                              additive=add),
            "x0": torch.ones(c["nx"] * c["ny"] * c["nz"], device=DEV)}


def run(state):
    c = state["c"]
    if c["kind"] == "osem":
        return state["run"].run(c["iters"], state["x0"])
    if c["kind"] == "project":
        if c["op"] == "forward":
            return state["p"].forwardProject(state["x"], 1)
        return state["p"].backwardProject(state["y"], 1)
    if c["kind"] == "ct":
        if c["op"] == "forward":
            return state["p"].forwardProject(state["x"], 1)
        return state["p"].backwardProject(state["y"], 1)
    if c["kind"] == "frames":
        r = state["run"]
        r.x.fill_(1.0)
        r.step(1, rays_per_block=128, frames_per_tile=2)
        return r.x
    net = state["net"]
    net.zero_grad()
    out = net.forward(state["image"], 1.0)
    loss = net.loss(state["target"], state["mask"], 1.0)
    net.backward(net.act["gout"])
    return {"out": out, "loss": loss, **net.g}


def _frame_activities(c, seed):
    rng = random.Random(seed + 5)
    rates = [(rng.uniform(0.05, 0.5), rng.uniform(0.5, 2.0)) for _ in range(8)]
    return [[a * (1.0 - math.exp(-r * (f + 1))) for r, a in rates] for f in range(c["frames"])]


def _ratio_data(c, seed):
    """What a backprojection meets: measured / expected ratios of the subset's LORs, about one."""
    n_planes = len(_subset_planes(c, _planes(c).shape[0])[1])
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.poisson(torch.full((n_planes * c["ndist"] * c["nang"],), 8.0, device=DEV), generator=g) / 8.0 + 0.05


def _ct_ellipsoids(c, seed):
    return _ellipsoids(seed, min(c["nx"], c["ny"]) * c["voxel"], c["nz"] * c["voxel"], 12, 0.002, 0.01)


def _ct_data(c, seed):
    """Line integrals of the subset's panels with 1% noise, detector row fastest."""
    x, uv = _ct_tables(c)
    k = _ct_subset(c)
    x, uv = torch.as_tensor(x[k], device=DEV), torch.as_tensor(uv[k], device=DEV)
    i1 = torch.arange(c["rows"], device=DEV) - c["rows"] / 2 + 0.5
    i2 = torch.arange(c["cols"], device=DEV) - c["cols"] / 2 + 0.5
    s = [x[:, j, None, None] for j in range(3)]
    d = (x[:, 3, None, None] + uv[:, 0, None, None] * i1, x[:, 4, None, None] + uv[:, 1, None, None] * i1,
         x[:, 5, None, None] + c["pixel"] * i2[None, :, None])
    v = [a - b for a, b in zip(d, s)]
    out = torch.zeros((len(k), c["cols"], c["rows"]), device=DEV)
    for ell in _ct_ellipsoids(c, seed):
        out += ell[6] * _chords(s, v, ell)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 3)
    out += 0.01 * out.max() * torch.randn(out.shape, device=DEV, generator=g)
    return out.reshape(-1).contiguous()


# ---- necessary work ------------------------------------------------------------------------------------------
def _crossings(c, planes):
    """(LORs, voxel intersections) of the given [zs, zd] planes: boundary crossings inside the image box."""
    xy = _ring_xy(c).astype(np.float64)
    h = c["fov"] / 2
    v = xy[:, 2:] - xy[:, :2]
    with np.errstate(divide="ignore", invalid="ignore"):
        ta, tb = (-h - xy[:, :2]) / v, (h - xy[:, :2]) / v
    t0 = np.nanmax(np.minimum(ta, tb), 1).clip(0, 1)
    t1 = np.nanmin(np.maximum(ta, tb), 1).clip(0, 1)
    f = np.maximum(t1 - t0, 0)
    n2 = np.where(f > 0, 1 + f * (np.abs(v[:, 0]) * c["nx"] / c["fov"] + np.abs(v[:, 1]) * c["ny"] / c["fov"]), 0).sum()
    dz = np.abs(planes[:, 1] - planes[:, 0]).astype(np.float64).sum() * c["nz"] / c["axial"]
    return len(planes) * len(xy), float(len(planes) * n2 + f.sum() * dz)


def work(case):
    c = case
    if c["kind"] == "unet":
        dims = [(-(-c["nz"] // 4) * 4 >> l) * (c["ny"] >> l) * (c["nx"] >> l) for l in range(3)]
        lev = {"e1a": 0, "e1b": 0, "e2a": 1, "e2b": 1, "bta": 2, "btb": 2, "d2a": 1, "d2b": 1, "d1a": 0, "d1b": 0}
        macs = sum(27 * dims[lev[n]] * i * o for n, i, o in LAYERS)
        first = 27 * dims[0] * 16 * 16
        # forward, weight gradient and (but for the first layer) data gradient; the activations once each way
        return {"bytes": 4.0 * dims[0] * 4 + 2 * 2 * sum(dims[lev[n]] * o for n, _, o in LAYERS),
                "flops": 2.0 * (3 * macs - first)}
    if c["kind"] == "ct":
        px = float(len(_ct_subset(c)) * c["rows"] * c["cols"])
        vox = float(c["nx"] * c["ny"] * c["nz"])
        # forward: an area difference of four table taps per pixel and slab; backward: per voxel and view
        flops = 8.0 * px * (c["nx"] + c["ny"]) / 2 if c["op"] == "forward" else 8.0 * vox * len(_ct_subset(c))
        return {"bytes": 4.0 * (px + vox), "flops": flops}
    vox = float(c["nx"] * c["ny"] * c["nz"])
    planes = _planes(c)
    if c["kind"] in ("project", "frames"):
        lors, cr = _crossings(c, planes[_subset_planes(c, len(planes))[1]])
        if c["kind"] == "project":
            return {"bytes": 4.0 * (lors + vox), "flops": 2.0 * float(cr)}
        hit = min(1.0, c["counts"] / (len(planes) * c["ndist"] * c["nang"]))
        return {"bytes": 4.0 * (c["frames"] * (lors + 2 * vox) + vox), "flops": 2.0 * c["frames"] * cr * (1 + hit)}
    lors, cr = _crossings(c, planes)
    bins = max(c["tof"], 1)
    if c["projector"] == 2:
        cr *= 1.4      # voxels of a 2.5 mm tube per voxel on its axis
    it = c["iters"]
    # per iteration forward and back projection, in the first one the sensitivity too; images per subset step
    return {"bytes": 4.0 * it * (bins * lors + 3 * vox * c["subsets"]), "flops": 2.0 * bins * cr * (2 * it + 1)}


def tolerance(case):
    # about four times what the start shows against the 64-bit results
    c = case
    if c["kind"] == "unet":
        return {"rel": 4e-2}         # bf16 activations and gradients through ten layers and their ReLU masks (1.7e-2)
    if c["kind"] == "ct":
        return {"rel": 1e-3}         # differences of 32-bit summed-area tables (2e-4 to 3.3e-4)
    if c["kind"] == "project":
        return {"rel": 2e-5}         # the 32-bit walk (the few LORs that it drops at the image's corners aside)
    return {"rel": 6e-5}             # the same walk through several multiplicative updates (2e-6 to 1.6e-5)


# ---- exact results ---------------------------------------------------------------------------------------------
def _f64(a):
    return torch.as_tensor(np.asarray(a), device=DEV).double()


def _siddon(src, dst, n, size):
    """Voxel indices and lengths [rays, crossings] (64-bit) of the segments src -> dst through the box."""
    v = dst - src
    L = v.norm(dim=1)
    ts, lo, hi = [], None, None
    for a in range(src.shape[1]):
        planes = torch.arange(n[a] + 1, device=DEV, dtype=torch.float64) * (size[a] / n[a]) - size[a] / 2
        va = torch.where(v[:, a].abs() < 1e-12, torch.full_like(v[:, a], 1e-12), v[:, a])
        t = (planes[None] - src[:, a, None]) / va[:, None]
        l, h = torch.minimum(t[:, 0], t[:, -1]), torch.maximum(t[:, 0], t[:, -1])
        lo = l if lo is None else torch.maximum(lo, l)
        hi = h if hi is None else torch.minimum(hi, h)
        ts.append(t)
    lo, hi = lo.clamp(0, 1), hi.clamp(0, 1)
    hi = torch.maximum(lo, hi)
    t = torch.cat(ts, 1)
    t = torch.minimum(torch.maximum(t, lo[:, None]), hi[:, None]).sort(1)[0]
    ln = (t[:, 1:] - t[:, :-1]) * L[:, None]
    mid = (t[:, 1:] + t[:, :-1]) / 2
    idx, stride = torch.zeros_like(mid, dtype=torch.int64), 1
    for a in range(src.shape[1]):
        q = (src[:, a, None] + mid * v[:, a, None] + size[a] / 2) / (size[a] / n[a])
        idx += q.floor().clamp(0, n[a] - 1).long() * stride
        stride *= n[a]
    return idx, ln, L


class _Rays3D:
    """64-bit Siddon projections of the LORs of a plane list, traced in chunks."""

    def __init__(self, c, planes):
        self.c = c
        self.n, self.size = (c["nx"], c["ny"], c["nz"]), (c["fov"], c["fov"], c["axial"])
        self.xy = _f64(_ring_xy(c))
        self.z = _f64(_planes(c)[planes])

    def chunks(self, bins=None):
        xy = self.xy if bins is None else self.xy[bins]
        step = max(1, 120000 // xy.shape[0])
        for p0 in range(0, self.z.shape[0], step):
            z = self.z[p0:p0 + step]
            k, m = z.shape[0], xy.shape[0]
            src = torch.cat([xy[:, :2].repeat(k, 1), z[:, 0].repeat_interleave(m)[:, None]], 1)
            dst = torch.cat([xy[:, 2:].repeat(k, 1), z[:, 1].repeat_interleave(m)[:, None]], 1)
            yield slice(p0 * m, (p0 + k) * m), _siddon(src, dst, self.n, self.size)


def _rdp(u, n, gamma, eps):
    """Relative difference prior gradient, 6 neighbours, zero outside (the update kernel's formula)."""
    x = torch.nn.functional.pad(u.reshape(n[2], n[1], n[0]), (1, 1, 1, 1, 1, 1))
    c = x[1:-1, 1:-1, 1:-1]
    out = torch.zeros_like(c)
    for a in range(3):
        for o in (0, 2):
            sl = [slice(1, -1)] * 3
            sl[a] = slice(o, x.shape[a] - 2 + o)
            w = x[tuple(sl)]
            d = c - w
            den = c + w + gamma * d.abs()
            out += torch.nan_to_num(d * (gamma * d.abs() + c + 3 * w + eps * eps) / (den * den + eps))
    return out.reshape(-1)


def _em(c, x, rhs, S):
    if c["beta"]:
        xn = x / (S + c["beta"] * _rdp(x, (c["nx"], c["ny"], c["nz"]), 2.0, EPPS)) * rhs
    else:
        xn = x / S * (rhs + EPPS)
    return xn.clamp_min(EPPS)


def _exact_osem3d(c, seed):
    y, _ = _pet_counts(c, seed)
    parts = _subset_order(c, y)
    rays = _Rays3D(c, np.arange(_planes(c).shape[0]))
    x = torch.ones(c["nx"] * c["ny"] * c["nz"], dtype=torch.float64, device=DEV)
    for k in range(c["subsets"]):
        bins = torch.arange(c["nang"] * c["ndist"], device=DEV).reshape(c["nang"], c["ndist"])[k::c["subsets"]].reshape(-1)
        rhs, S = torch.zeros_like(x), torch.zeros_like(x)
        for sl, (idx, ln, L) in rays.chunks(bins):
            w = ln / L[:, None]
            r = parts[k][0, sl].double() / ((x[idx] * w).sum(1) + EPPS)
            rhs.index_add_(0, idx.reshape(-1), (w * r[:, None]).reshape(-1))
            S.index_add_(0, idx.reshape(-1), w.reshape(-1))
        x = _em(c, x, rhs, S.clamp_min(EPPS))
    return x


def _exact_plane_system(c):
    """Direct planes share one 2-D system: indices and weights [bins, K] and, with TOF, the share of every TOF
    bin [bins, K, TOF bins]."""
    n, size = (c["nx"], c["ny"]), (c["fov"], c["fov"])
    xy = _f64(_ring_xy(c))
    idx, ln, L = _siddon(xy[:, :2], xy[:, 2:], n, size)
    lor = 1.0 / L
    if c["atten"]:
        mu = _f64(_mu_image(c))[: c["nx"] * c["ny"]]
        lor = lor * torch.exp(-(ln * mu[idx]).sum(1))
    if c["projector"] == 1:
        if not c["tof"]:
            return idx, ln * lor[:, None], None
        sigma, cen = _tof_tables(c)
        sigma, cen = float(sigma), _f64(cen)
        entry = _entry(xy, size) * L
        D = (entry - L / 2)[:, None] + torch.cat([torch.zeros_like(ln[:, :1]), ln.cumsum(1)[:, :-1]], 1)
        # LORs along an image axis measure the distance down the axis (up it where the step across is negative)
        v = xy[:, 2:] - xy[:, :2]
        flip = torch.ones_like(L)
        for a in range(2):
            flip = torch.where(v[:, 1 - a].abs() < 1e-8, -torch.sign(v[:, a]) * torch.copysign(flip.abs(), v[:, 1 - a]), flip)
        w = torch.zeros(ln.shape + (c["tof"],), dtype=torch.float64, device=DEV)
        for q, m in ((0.0, 1.0), (1 / 3, 2.0), (2 / 3, 2.0), (1.0, 1.0)):
            for b in range(c["tof"]):
                w[:, :, b] += m * torch.exp(-0.5 * (((D + q * ln) * flip[:, None] - cen[b]) / sigma) ** 2)
        w *= 0.3989422804014327 / sigma * (ln / 3)[:, :, None]
        w /= w.sum(2).clamp_min(EPPS)[:, :, None]
        return idx, ln * lor[:, None], w
    # every voxel of the slice whose centre lies within 0.99 widths of the line weighs 1 - d / width
    width = 2.5
    gx = (torch.arange(n[0], device=DEV, dtype=torch.float64) + 0.5) * (size[0] / n[0]) - size[0] / 2
    gy = (torch.arange(n[1], device=DEV, dtype=torch.float64) + 0.5) * (size[1] / n[1]) - size[1] / 2
    cx, cy = gx.repeat(n[1]), gy.repeat_interleave(n[0])
    v = (xy[:, 2:] - xy[:, :2]) / L[:, None]
    keep, K = [], 0
    hit = ln.sum(1) > 0
    for b0 in range(0, xy.shape[0], 2048):
        s, u = xy[b0:b0 + 2048, :2], v[b0:b0 + 2048]
        d = ((cx - s[:, :1]) * u[:, 1:] - (cy - s[:, 1:]) * u[:, :1]).abs()
        wgt = torch.where((d < 0.99 * width) & hit[b0:b0 + 2048, None], 1 - d / width, 0.0)
        K = max(K, int((wgt > 0).sum(1).max()))
        keep.append(wgt.topk(min(5 * max(n), n[0] * n[1]), dim=1))
    idx = torch.cat([k.indices[:, :K] for k in keep])
    return idx, torch.cat([k.values[:, :K] for k in keep]) * (lor * L)[:, None], None     # not divided by the length


def _entry(xy, size):
    """Parameter at which the lines enter the image."""
    out = None
    for a in range(2):
        v = xy[:, 2 + a] - xy[:, a]
        v = torch.where(v.abs() < 1e-12, torch.full_like(v, 1e-12), v)
        ta, tb = (-size[a] / 2 - xy[:, a]) / v, (size[a] / 2 - xy[:, a]) / v
        t = torch.minimum(ta, tb)
        out = t if out is None else torch.maximum(out, t)
    return out


def _exact_osem2d(c, seed):
    y, mean = _pet_counts(c, seed)
    add = 0.2 * mean[0] + 0.05 * mean.mean() if c["randoms"] else None
    add = None if add is None else add.double()
    idx, w, tw = _exact_plane_system(c)
    nyx, nz = c["nx"] * c["ny"], c["nz"]
    x = torch.ones((nz, nyx), dtype=torch.float64, device=DEV)
    sens = torch.zeros(nyx, dtype=torch.float64, device=DEV)
    sens.index_add_(0, idx.reshape(-1), (w if tw is None else w * tw.sum(2)).reshape(-1))
    for _ in range(c["iters"]):
        for planes in _subset_planes(c, nz):
            S = torch.full_like(x, EPPS)
            rhs = torch.zeros_like(x)
            for z in planes:
                S[z] = sens.clamp_min(EPPS)
                xg = x[z][idx] * w
                extra = 0.0 if add is None else add[z]
                if tw is None:
                    r = y[0, z].double() / (xg.sum(1) + EPPS + extra)
                    val = w * r[:, None]
                else:
                    val = torch.zeros_like(w)
                    for b in range(c["tof"]):
                        r = y[b, z].double() / ((xg * tw[:, :, b]).sum(1) + EPPS + extra)
                        val += w * tw[:, :, b] * r[:, None]
                rhs[z].index_add_(0, idx.reshape(-1), val.reshape(-1))
            x = _em(c, x.reshape(-1), rhs.reshape(-1), S.reshape(-1)).reshape(nz, nyx)
    return x.reshape(-1)


def _exact_project(c, seed):
    planes = np.asarray(_subset_planes(c, _planes(c).shape[0])[1])
    rays = _Rays3D(c, planes)
    if c["op"] == "forward":
        x = _image(_ellipsoids(seed, c["fov"], c["axial"]), 0.1, rays.n, rays.size).double()
        return torch.cat([(x[idx] * ln).sum(1) / L for _, (idx, ln, L) in rays.chunks()])
    y = _ratio_data(c, seed).double()
    out = torch.zeros(c["nx"] * c["ny"] * c["nz"], dtype=torch.float64, device=DEV)
    for sl, (idx, ln, L) in rays.chunks():
        out.index_add_(0, idx.reshape(-1), (ln * (y[sl] / L)[:, None]).reshape(-1))
    return out


def _exact_frames(c, seed):
    y, _ = _pet_counts(c, seed, _frame_activities(c, seed))
    planes = _subset_planes(c, y.shape[1])[1]
    yk = y[:, planes].reshape(y.shape[0], -1)
    del y
    rays = _Rays3D(c, np.asarray(planes))
    S = torch.zeros(c["nx"] * c["ny"] * c["nz"], dtype=torch.float64, device=DEV)
    rhs = torch.zeros((yk.shape[0], S.numel()), dtype=torch.float64, device=DEV)
    for sl, (idx, ln, L) in rays.chunks():
        w = ln / L[:, None]
        S.index_add_(0, idx.reshape(-1), w.reshape(-1))
        yhat = w.sum(1) + EPPS         # the step starts from an image of ones
        for f in range(yk.shape[0]):
            hit = yk[f, sl] != 0
            rhs[f].index_add_(0, idx[hit].reshape(-1), (w[hit] * (yk[f, sl][hit].double() / yhat[hit])[:, None]).reshape(-1))
    return ((rhs + EPPS) / S.clamp_min(EPPS)).clamp_min(EPPS)


def _lerp_rows(T, pos):
    """Linear interpolation of T along its last axis at pos (clamped to the ends)."""
    f = pos.floor()
    a = pos - f
    i0, i1 = f.clamp(0, T.shape[-1] - 1).long(), (f + 1).clamp(0, T.shape[-1] - 1).long()
    return (1 - a) * torch.gather(T, -1, i0) + a * torch.gather(T, -1, i1)


def _exact_ct_forward(c, seed):
    n, vs = (c["nx"], c["ny"], c["nz"]), c["voxel"]
    size = tuple(k * vs for k in n)
    vol = _image(_ct_ellipsoids(c, seed), 0.004, n, size).double().reshape(n[2], n[1], n[0])
    tab = torch.nn.functional.pad(vol.cumsum(0), (0, 0, 0, 0, 1, 0))       # prefix along z
    x, uv = _ct_tables(c)
    k = _ct_subset(c)
    x, uv = _f64(x[k]), _f64(uv[k])
    i1 = torch.arange(c["rows"], device=DEV, dtype=torch.float64) - c["rows"] / 2 + 0.5
    edge = (torch.arange(c["cols"] + 1, device=DEV, dtype=torch.float64) - c["cols"] / 2) * c["pixel"]
    first = (torch.arange(c["cols"], device=DEV) // 8 * 8 - c["cols"] / 2 + 0.5) * c["pixel"]
    out = torch.zeros((len(k), c["cols"], c["rows"]), dtype=torch.float64, device=DEV)
    for v in range(len(k)):
        s, d, u = x[v, :3], x[v, 3:], uv[v]
        ydir = bool(s[0].abs() <= s[1].abs())
        a, b = (0, 1) if ydir else (1, 0)          # across, along
        slabs = tab.permute(1, 2, 0) if ydir else tab.permute(2, 1, 0)     # [slab, across, z]
        slabs = torch.nn.functional.pad(slabs.cumsum(1), (0, 0, 1, 0))
        pc = [d[j] + i1 * u[j] for j in range(2)]
        lo = (pc[a] + u[a] / 2 - s[a]) / (pc[b] + u[b] / 2 - s[b])
        hi = (pc[a] - u[a] / 2 - s[a]) / (pc[b] - u[b] / 2 - s[b])
        vv = (torch.arange(n[b], device=DEV, dtype=torch.float64) + 0.5) * vs - size[b] / 2 - s[b]
        tl = torch.minimum(vv[:, None] * lo, vv[:, None] * hi)             # [slab, row]
        tr = torch.maximum(vv[:, None] * lo, vv[:, None] * hi)
        zr = (edge[None] + d[2] - s[2]) / (pc[b] - s[b])[:, None]          # [row, edge]
        ex, ey = pc[0] - s[0], pc[1] - s[1]
        ez = first[:, None] + d[2] - s[2]                                  # the cosine is the column group's
        cosv = (ey if ydir else ex).abs()[None] / torch.sqrt(ex[None] ** 2 + ey[None] ** 2 + ez ** 2)
        for j in range(n[b]):
            T = slabs[j].t()                                               # [z, across]
            g = _lerp_rows(T, ((tr[j] + s[a] + size[a] / 2) / vs)[None].expand(T.shape[0], -1)) - \
                _lerp_rows(T, ((tl[j] + s[a] + size[a] / 2) / vs)[None].expand(T.shape[0], -1))
            ze = vv[j] * zr
            h = _lerp_rows(g.t().contiguous(), (ze + s[2] + size[2] / 2) / vs)
            area = ((tr[j] - tl[j])[:, None] * (ze[:, 1:] - ze[:, :-1])).abs()
            out[v] += ((h[:, 1:] - h[:, :-1]) / area).abs().t()
        out[v] *= vs ** 3 / cosv
    return out.reshape(-1)


def _exact_ct_backward(c, seed):
    n, vs = (c["nx"], c["ny"], c["nz"]), c["voxel"]
    size = tuple(k * vs for k in n)
    y = _ct_data(c, seed).double().reshape(-1, c["cols"], c["rows"])
    tab = torch.nn.functional.pad(y.cumsum(1).cumsum(2), (1, 0, 1, 0))
    x, uv = _ct_tables(c)
    k = _ct_subset(c)
    x, uv = _f64(x[k]), _f64(uv[k])
    vx = (torch.arange(n[0], device=DEV, dtype=torch.float64) + 0.5) * vs - size[0] / 2
    vy = (torch.arange(n[1], device=DEV, dtype=torch.float64) + 0.5) * vs - size[1] / 2
    vz = (torch.arange(n[2], device=DEV, dtype=torch.float64) + 0.5) * vs - size[2] / 2
    X, Y = vx[None, :].expand(n[1], n[0]).reshape(-1), vy[:, None].expand(n[1], n[0]).reshape(-1)
    out = torch.zeros((n[2], n[0] * n[1]), dtype=torch.float64, device=DEV)
    for v in range(len(k)):
        s, d, u = x[v, :3], x[v, 3:], uv[v]
        ydir = bool(s[0].abs() <= s[1].abs())
        un = u / u.norm()
        nrm = torch.stack([un[1], -un[0]])
        dist = (d[0] - s[0]) * nrm[0] + (d[1] - s[1]) * nrm[1]
        pos = []
        sgn = 1.0 if float(s[1] if ydir else s[0]) > 0 else -1.0
        for o in (-1.0, 1.0):       # the two faces of the voxel seen across the view, with their own scale
            if ydir:
                px, py = X + o * sgn * vs / 2 - s[0], Y - s[1]
            else:
                px, py = X - s[0], Y - o * sgn * vs / 2 - s[1]
            t = dist / (px * nrm[0] + py * nrm[1])
            col = (t[None] * (vz[:, None] + o * vs / 2 - s[2]) + s[2] - d[2]) / c["pixel"] + c["cols"] / 2
            row = ((t * px + s[0] - d[0]) * un[0] + (t * py + s[1] - d[1]) * un[1]) / c["pixel"] + c["rows"] / 2
            pos.append((row, col))
        r0, r1 = torch.minimum(pos[0][0], pos[1][0]), torch.maximum(pos[0][0], pos[1][0])
        c0, c1 = torch.minimum(pos[0][1], pos[1][1]), torch.maximum(pos[0][1], pos[1][1])

        def tap(r, q):              # r [xy], q [z, xy]
            fr, fq = r.floor(), q.floor()
            ar, aq = r - fr, q - fq
            R = [(fr + o).clamp(0, c["rows"]).long() for o in (0, 1)]
            Q = [(fq + o).clamp(0, c["cols"]).long() * (c["rows"] + 1) for o in (0, 1)]
            T = tab[v].reshape(-1)
            return (1 - aq) * ((1 - ar) * T[Q[0] + R[0]] + ar * T[Q[0] + R[1]]) + \
                aq * ((1 - ar) * T[Q[1] + R[0]] + ar * T[Q[1] + R[1]])

        area = tap(r1, c1) - tap(r0, c1) - tap(r1, c0) + tap(r0, c0)
        dxv, dyv, dzv = X - s[0], Y - s[1], (vz - s[2])[:, None]
        out += area * vs * torch.sqrt((dxv ** 2 + dyv ** 2)[None] + dzv ** 2) / (dyv if ydir else dxv).abs()
    return out.reshape(-1)


def _exact_unet(c, seed):
    par = {k: _f64(v).requires_grad_(True) for k, v in _unet_params(seed).items()}
    image, target = (t.double() for t in _unet_images(c, seed))
    D, H, W = -(-c["nz"] // 4) * 4, c["ny"], c["nx"]

    def conv(x, name):
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        d, h, w = x.shape[:3]
        out = par[name + ".b"]
        for t in range(27):
            z, y, q = t // 9, t // 3 % 3, t % 3
            out = out + p[z:z + d, y:y + h, q:q + w] @ par[name + ".w"][t].t()
        return torch.relu(out)

    def pool(x):
        d, h, w, ch = x.shape
        return x.reshape(d // 2, 2, h // 2, 2, w // 2, 2, ch).mean((1, 3, 5))

    def up(x):
        return x.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)

    full = torch.zeros(D * H * W, dtype=torch.float64, device=DEV)
    full[: image.numel()] = image
    x0 = torch.nn.functional.pad(full.reshape(D, H, W, 1), (0, 15))
    s1 = conv(conv(x0, "e1a"), "e1b")
    s2 = conv(conv(pool(s1), "e2a"), "e2b")
    b3 = conv(conv(pool(s2), "bta"), "btb")
    d2 = conv(conv(torch.cat([up(b3), s2], 3), "d2a"), "d2b")
    d1 = conv(conv(torch.cat([up(d2), s1], 3), "d1a"), "d1b")
    out = full + par["head.b"] + (d1 @ par["head.w"]).reshape(-1)
    loss = ((out[: target.numel()] - target) ** 2).sum() / target.numel()
    loss.backward()
    return {"out": out.detach(), "loss": loss.detach().reshape(1), **{k: v.grad for k, v in par.items()}}


def exact(case, seed):
    c = case
    if c["kind"] == "unet":
        return _exact_unet(c, seed)
    if c["kind"] == "ct":
        return _exact_ct_forward(c, seed) if c["op"] == "forward" else _exact_ct_backward(c, seed)
    if c["kind"] == "project":
        return _exact_project(c, seed)
    if c["kind"] == "frames":
        return _exact_frames(c, seed)
    if c["projector"] == 4:
        return None    # its first sample lies on the image's face: rounding decides the voxel that it updates
    return _exact_osem3d(c, seed) if c["rings"] else _exact_osem2d(c, seed)
