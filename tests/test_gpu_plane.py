"""Subset iterations of direct-plane sinograms from the shared 2-D system's lists (plane.hip) against the same
iterations through the one-lane-per-LOR kernels (omg_geom_desc.reserved[0]).

Both sum the same 32-bit products; the lists sum the backprojection in double, the other kernels in 32-bit
atomics over at most ~400 LORs per voxel, so the images agree within about 400 * 2^-24 / sqrt(400) = 1.2e-6 per
update; bar: 5e-6 relative L2 after two updates. Plane counts of 1, 2, 3, 5 and 9 per call cover every lane
grouping and a second chunk of planes; images that are odd, non-square and smaller than one block; a plane
outside the image; two planes of one slice (where the lists do not apply); every register group of TOF bins; the
interpolation projector's far-face samples, which carry into the next slice.
"""
import ctypes as C

import numpy as np
import pytest

from omega_amd import _lib, geometry as G
from tests.hip_helpers import list_calls, make_geom, ptr, rel_l2

pytestmark = pytest.mark.gpu
EPPS = 1e-5


def _scanner(nx, ny, nz, n_radial, n_angles, extra_z=(), dz=2.5):
    fov = 2.5 * max(nx, ny)
    grid = G.Grid.from_fov(nx, ny, nz, fov, fov, dz * nz)
    x = G.ring_sinogram_xy(n_radial, n_angles, fov / n_radial, 1.25 * fov)
    z = G.direct_planes_z(grid)
    if extra_z:
        z = np.concatenate([z, np.repeat(np.asarray(extra_z, np.float32), 2)])
    return grid, x, z


def _iterate(geom, grid, first, planes, per, meas, add, beta, seed):
    import torch
    rng = np.random.default_rng(seed)
    x = torch.from_numpy((rng.random(grid.N) + 0.5).astype(np.float32)).cuda()
    S = torch.zeros(grid.N, device="cuda")
    for sens in (1, 0):
        _lib.call("omg_osem_subset_iteration_ex", geom.handle, first, planes * per, ptr(x), ptr(meas), ptr(add),
                  ptr(S), sens, EPPS, beta, 2.0, 1, None)
    torch.cuda.synchronize()
    return x.cpu().numpy(), S.cpu().numpy()


def _entries(grid, x, z, n_radial, n_angles):
    """Entries of the row lists of one plane: eight rows side by side, each padded to the longest and to a multiple of 8."""
    import torch
    per = n_radial * n_angles
    geom, counts = make_geom(grid, x, z, n_radial, n_angles), torch.zeros(per, dtype=torch.int32, device="cuda")
    _lib.call("omg_siddon_trace", geom.handle, 0, per, ptr(counts), None, None, None, None)
    longest = np.pad(counts.cpu().numpy(), (0, -per % 8)).reshape(-1, 8).max(axis=1)
    return int((-(-longest // 8) * 64).sum())


def _lists_fit(grid, x, z, n_radial, n_angles, mib, tof):
    """Whether an iteration on one plane runs from lists within ``mib``."""
    import torch
    per = n_radial * n_angles
    geom = make_geom(grid, x, z, n_radial, n_angles, tof=tof, tube_budget_mib=mib)
    img, S, meas = torch.ones(grid.N, device="cuda"), torch.zeros(grid.N, device="cuda"), torch.ones(per * tof[0], device="cuda")
    _lib.call("omg_osem_subset_iteration_ex", geom.handle, 0, per, ptr(img), ptr(meas), None, ptr(S), 1, EPPS, 0.0, 2.0, 1,
              None)
    torch.cuda.synchronize()
    return list_calls(geom) == (1, 0)


def _compare(grid, x, z, n_radial, n_angles, first, planes, bins=1, beta=0.0, add=False, lists=True, **kw):
    import torch
    per = n_radial * n_angles
    rng = np.random.default_rng(planes + grid.Nx)
    meas = torch.from_numpy(rng.poisson(3.0, planes * per * bins).astype(np.float32)).cuda()
    a = torch.from_numpy((rng.random(planes * per) + 0.1).astype(np.float32)).cuda() if add else None
    out = []
    for generic in (False, True):
        geom = make_geom(grid, x, z, n_radial, n_angles, generic=generic, **kw)
        out.append(_iterate(geom, grid, first, planes, per, meas, a, beta, 3))
        out.append(_iterate(geom, grid, first, planes, per, meas, a, beta, 3)) if not generic else None
        assert list_calls(geom) == ((0 if generic or not lists else 4), 0)
    (xa, Sa), (xb, _), (xg, Sg) = out
    if lists:                       # the other kernels add with atomics
        assert np.array_equal(xa, xb)   # the lists have a fixed order
    e, es = rel_l2(xa, xg), rel_l2(Sa, Sg)
    print(f"[plane] {grid.Nx}x{grid.Ny}x{grid.Nz} planes={planes} bins={bins} rel-L2 {e:.2e} sens {es:.2e}", flush=True)
    assert e < 5e-6 and es < 5e-6
    return xa


@pytest.mark.parametrize("nx,ny,nz,n_radial,n_angles", [(32, 32, 11, 32, 40), (21, 34, 10, 29, 27), (5, 5, 9, 7, 9)])
@pytest.mark.parametrize("planes", [1, 2, 3, 5, 9])
def test_siddon(cuda, nx, ny, nz, n_radial, n_angles, planes):
    grid, x, z = _scanner(nx, ny, nz, n_radial, n_angles)
    norm = np.random.default_rng(0).random(n_radial * n_angles * nz).astype(np.float32) + 0.5
    _compare(grid, x, z, n_radial, n_angles, 0 if planes == 9 else 1, planes, add=planes % 2 == 1,
             beta=0.01 if planes > 2 else 0.0, norm=norm, global_factor=0.9)


def test_plane_outside_and_shared_slice(cuda):
    grid, x, z = _scanner(20, 20, 6, 24, 21, extra_z=(100.0, 1.25))   # beyond the image; slice 3's centre again
    _compare(grid, x, z, 24, 21, 3, 4)      # planes 3, 4, 5 and the one outside
    import torch
    per = 24 * 21
    geom = make_geom(grid, x, z, 24, 21)
    gen = make_geom(grid, x, z, 24, 21, generic=True)
    meas = torch.ones(8 * per, device="cuda")
    a = _iterate(geom, grid, 0, 8, per, meas, None, 0.0, 5)[0]
    assert list_calls(geom) == (0, 0)
    b = _iterate(gen, grid, 0, 8, per, meas, None, 0.0, 5)[0]
    assert rel_l2(a, b) < 5e-6


@pytest.mark.parametrize("bins,planes", [(3, 2), (8, 9), (13, 1), (17, 5), (23, 3), (32, 2), (33, 2)])
def test_tof(cuda, bins, planes):
    grid, x, z = _scanner(22, 19, 10, 24, 21)
    sigma = G.tof_sigma(300e-12)
    centres = np.linspace(-40.0, 40.0, bins).astype(np.float32)
    atten = np.full(grid.N, 0.004, np.float32)
    _compare(grid, x, z, 24, 21, 1, planes, bins=bins, add=True, lists=bins <= 32, tof=(bins, sigma, centres, EPPS),
             atten=atten, atten_mode=1)


@pytest.mark.parametrize("n,flags,planes", [(32, 3, 5), (19, 3, 2), (20, 1, 9)])
def test_orthogonal(cuda, n, flags, planes):
    grid, x, z = _scanner(n, n, 10, 24, 20)
    _compare(grid, x, z, 24, 20, 0, planes, projector_type=2, orth_width=2.4, orth_flags=flags,
             norm=np.random.default_rng(1).random(24 * 20 * 10).astype(np.float32) + 0.5)


@pytest.mark.parametrize("nx,ny,dl,atten", [(32, 32, 2.5, False), (21, 34, 1.7, True), (16, 16, -2.5, False)])
@pytest.mark.parametrize("planes", [1, 4, 9])
def test_interpolation(cuda, nx, ny, dl, atten, planes):
    grid, x, z = _scanner(nx, ny, 10, 24, 20)
    kw = dict(atten=np.full(grid.N, 0.004, np.float32), atten_mode=1) if atten else {}
    _compare(grid, x, z, 24, 20, 0, planes, projector_type=4, interp=(dl, 0.0), beta=0.01, **kw)


def test_lists_off(cuda):
    """A negative budget keeps no lists."""
    grid, x, z = _scanner(32, 32, 11, 32, 40)
    _compare(grid, x, z, 32, 40, 0, 5, lists=False, tube_budget_mib=-1)


@pytest.mark.parametrize("descending", [False, True])
@pytest.mark.parametrize("tof", [False, True])
def test_rows_past_the_slice(cuda, descending, tof):
    """Ny > Nx and LORs along x: those step rows by Ny, so their voxels run on into the next slices and, from the last
    ones, past the image. Whichever plane comes first, the result is the other kernels'."""
    grid, x, z = _scanner(21, 34, 10, 29, 28)
    z = z.reshape(-1, 2)[::-1].copy() if descending else z
    kw = dict(tof=(5, G.tof_sigma(300e-12), np.linspace(-40.0, 40.0, 5).astype(np.float32), EPPS), bins=5) if tof else {}
    _compare(grid, x, z, 29, 28, 2, 5, lists=not tof, beta=0.01, **kw)
    _compare(grid, x, z, 29, 28, 0, 9, lists=not tof, **kw)
    grid, x, z = _scanner(9, 34, 10, 29, 28)          # over more than one slice
    _compare(grid, x, z[::-1] if descending else z, 29, 28, 1, 8, lists=not tof, **kw)


def test_captured_iterations(cuda):
    """Iterations captured on a handle with lists: one whose work memory later calls outgrow, and one that would have to
    grow it while capturing. Replays between eager work give what the same iterations give eagerly."""
    import torch
    grid, x, z = _scanner(22, 19, 10, 24, 21)
    per, bins = 24 * 21, 5
    geom = make_geom(grid, x, z, 24, 21,
                     tof=(bins, G.tof_sigma(300e-12), np.linspace(-40.0, 40.0, bins).astype(np.float32), EPPS))
    meas = torch.poisson(torch.full((9 * per * bins,), 3.0, device="cuda"))
    side = torch.cuda.Stream()

    def iterate(img, S, planes, sens=1):
        _lib.call("omg_osem_subset_iteration_ex", geom.handle, 0, planes * per, ptr(img), ptr(meas), None, ptr(S), sens,
                  EPPS, 0.0, 2.0, 1, C.c_void_p(torch.cuda.current_stream().cuda_stream))

    start = torch.rand(grid.N, device="cuda") + 0.5
    iterate(start.clone(), torch.zeros(grid.N, device="cuda"), 1)      # lists, and work memory for one plane
    buf = [(torch.zeros(grid.N, device="cuda"), torch.zeros(grid.N, device="cuda")) for _ in range(2)]
    torch.cuda.synchronize()
    graphs = []
    for (img, S), planes in zip(buf, (1, 9)):                          # the second is captured tracing
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=side):
            iterate(img, S, planes)
    assert list_calls(geom) == (2, 0)
    for k in range(3):
        for (img, S), planes, graph in zip(buf, (1, 9), graphs):
            want, Sw = start.clone(), torch.zeros(grid.N, device="cuda")
            iterate(want, Sw, planes)                                  # outgrows the memory of the first graph
            img.copy_(start)
            S.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert rel_l2(img.cpu().numpy(), want.cpu().numpy()) < 5e-6
            assert rel_l2(S.cpu().numpy(), Sw.cpu().numpy()) < 5e-6


def test_budget_counts_work_memory(cuda):
    """17 TOF bins of 48 x 63 LORs: the budget holds the lists (92 bytes per entry, and the pixel lists) and an iteration's
    sums (32 bytes per entry)."""
    grid, x, z = _scanner(48, 48, 9, 48, 63)
    kw = dict(bins=17, tof=(17, G.tof_sigma(300e-12), np.linspace(-80.0, 80.0, 17).astype(np.float32), EPPS))
    sizes = [m for m in range(8, 33) if _lists_fit(grid, x, z, 48, 63, m, kw["tof"])]
    print(f"[plane] lists and work memory fit from {sizes[0]} MiB", flush=True)
    nent = _entries(grid, x, z, 48, 63)
    print(f"[plane] {nent} entries", flush=True)
    assert sizes == list(range(sizes[0], 33)) and sizes[0] << 20 > nent * (8 + 4 + 4 * 20 + 32)
    _compare(grid, x, z, 48, 63, 0, 9, lists=False, tube_budget_mib=sizes[0] - 1, **kw)


@pytest.mark.parametrize("dz,nz", [(2.027, 109), (2.425, 63), (3.27, 47), (1.775, 83), (2.4, 62)])
def test_orthogonal_slice_spacing(cuda, dz, nz):
    """Slices whose thickness is no short binary fraction: the planes' offsets from their slice centres differ by the
    rounding of the coordinates and of dz, and the lists are of one of them. A weight differs by
    at most spread / width (1e-4) where a voxel's centre lies on the LOR, and by less than 1e-7 from 0.1 mm on."""
    grid, x, z = _scanner(20, 20, nz, 24, 20, dz=dz)
    z = np.repeat((np.arange(nz) + 0.5) * dz - 0.5 * dz * nz, 2).astype(np.float32)
    f = np.float32
    tk = (np.abs(z[::2] - f(grid.bz)) / f(grid.dz)).astype(np.int32).astype(f)
    off = (f(grid.bz) + tk * f(grid.dz) + f(grid.dz) / f(2)) - z[::2]
    spread = float(off.max() - off.min())
    assert spread > 0
    print(f"[plane] {len(set(off.tolist()))} offsets over {spread:.1e} mm", flush=True)
    _compare(grid, x, z, 24, 20, nz - 9, 9, projector_type=2, orth_width=1.7, orth_flags=3)


def test_orthogonal_offsets_apart(cuda):
    """Planes that lie at different offsets by more than rounding keep lists of their own."""
    grid, x, z = _scanner(20, 20, 10, 24, 20)
    z = z + np.repeat(np.arange(10) * 1e-3, 2).astype(np.float32)
    _compare(grid, x, z, 24, 20, 0, 9, lists=False, projector_type=2, orth_width=1.7, orth_flags=3)
