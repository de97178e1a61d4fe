"""3-D sinograms by image columns (column.hip) against the one-lane-per-LOR kernels (omg_geom_desc.reserved[0]).

The forward projection adds the same 32-bit products in the same order, so it is compared bit for bit. The
backprojection adds the same products in 64-bit fixed point where the other kernels use 32-bit float atomics over at
most ~5e3 terms per voxel: 2^-24 sqrt(5e3) = 4e-6 relative L2; bar 2e-5. A length between two crossings carries the
rounding of their parameters, 2^-24 of a LOR of up to ~150 mm (1e-5 mm) each: the updated image is compared where the
sensitivity is at least 0.5 mm, so that a voxel's own error stays below the bar. Images of one, two and more than two
registers of slices per lane, odd, non-square and smaller than a tile; plane counts around the 64 of a wave, and below the 32 where
only the backprojection goes by columns; planes
far steeper than a voxel, outside the image, and leaving it through an end face.
"""
import ctypes as C

import numpy as np
import pytest

from omega_amd import _lib, geometry as G
from tests.hip_helpers import list_calls, make_geom, ptr, rel_l2

pytestmark = pytest.mark.gpu
EPPS = 1e-5
BAR = 2e-5


def _scanner(nx, ny, nz, n_radial, n_angles, planes, dz=2.5):
    fov = 2.5 * max(nx, ny)
    grid = G.Grid.from_fov(nx, ny, nz, fov, fov, dz * nz)
    x = G.ring_sinogram_xy(n_radial, n_angles, fov / n_radial, 1.25 * fov)
    rng = np.random.default_rng(planes)
    half = 0.5 * dz * nz
    z = rng.uniform(-half, half, (planes, 2))
    z[:: 5] = np.repeat(grid.centers()[2][rng.integers(0, nz, len(z[::5]))][:, None], 2, axis=1)   # direct
    z[1:: 7] *= 6.0                                                                                # through the end faces
    z[3] = (2.0 * half, 3.0 * half)                                                                # beside the image
    return grid, x, z.astype(np.float32)


def _run(geom, grid, first, n, img, y, meas):
    import torch
    out = torch.empty(n, device="cuda")
    _lib.call("omg_forward_project", geom.handle, first, n, ptr(img), ptr(out), None)
    back, S = torch.zeros(grid.N, device="cuda"), torch.zeros(grid.N, device="cuda")
    _lib.call("omg_backward_project", geom.handle, first, n, ptr(y), ptr(back), ptr(S), None)
    x, Sx = img.clone(), torch.zeros(grid.N, device="cuda")
    for sens in (1, 0):
        _lib.call("omg_osem_subset_iteration_ex", geom.handle, first, n, ptr(x), ptr(meas), None, ptr(Sx), sens, EPPS,
                  0.0, 2.0, 1, None)
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in (out, back, S, x, Sx)]


@pytest.mark.parametrize("nx,ny,nz,n_radial,n_angles,planes,first,dz", [
    (20, 20, 9, 24, 20, 32, 0, 2.5), (33, 21, 15, 29, 23, 63, 1, 2.5), (7, 5, 63, 11, 9, 64, 0, 2.5),
    (17, 18, 64, 19, 16, 65, 0, 1.0), (16, 32, 127, 20, 12, 40, 0, 0.7), (16, 16, 128, 20, 12, 70, 2, 0.6),
    (3, 3, 301, 8, 6, 129, 0, 0.3), (20, 18, 11, 24, 20, 12, 1, 2.5), (20, 18, 11, 24, 20, 31, 0, 2.5), (40, 40, 2, 32, 32, 130, 0, 9.0)])
def test_column(cuda, nx, ny, nz, n_radial, n_angles, planes, first, dz):
    import torch
    grid, x, z = _scanner(nx, ny, nz, n_radial, n_angles, planes + first, dz)
    n = planes * n_radial * n_angles
    rng = np.random.default_rng(1)
    norm = rng.random(n_radial * n_angles * (planes + first)).astype(np.float32) + 0.5
    up = lambda a: torch.from_numpy(a.astype(np.float32)).cuda()
    img, y, meas = up(rng.random(grid.N) + 0.5), up(rng.standard_normal(n)), up(rng.poisson(2.0, n))
    geoms = [make_geom(grid, x, z, n_radial, n_angles, generic=gen, norm=norm, global_factor=0.9) for gen in (False, True)]
    a, b = (_run(g, grid, first, n, img, y, meas) for g in geoms)
    assert [list_calls(g) for g in geoms] == [(0, 4 if planes >= 32 else 1), (0, 0)]
    seen = b[4] > 0.5
    assert seen.any()
    a[3], b[3] = a[3][seen], b[3][seen]
    e = [rel_l2(p, q) for p, q in zip(a, b)]
    print(f"[column] {nx}x{ny}x{nz} planes={planes} rel-L2 {e}", flush=True)
    assert np.array_equal(a[0], b[0])
    assert max(e[1:]) < BAR


@pytest.mark.parametrize("k", [1, 3, 8, 14, 21])
def test_ranges_built_together(cuda, k):
    """Index tables of k equal ranges, called from the middle on: up to 8 are built at the first call, more at the second
    in batches of 8. One range is not the same bins in every plane, and is traced."""
    import torch
    planes, per = 40, 21 * 16
    grid, x, z = _scanner(20, 20, 9, 21, 16, planes)
    b = per // k
    bins = np.random.default_rng(k).permutation(per)[:k * b].reshape(k, b)
    index = (np.arange(planes)[None, :, None] * per + bins[:, None, :]).astype(np.uint32)
    odd = k - 1
    index[odd, 7] = index[odd, 7][::-1]
    img, n = torch.rand(grid.N, device="cuda") + 0.5, planes * b
    out = []
    for gen in (False, True):
        g = make_geom(grid, x, z, 21, 16, meas_index=index.ravel(), generic=gen)
        y = torch.empty(k * n, device="cuda")
        back = torch.zeros(grid.N, device="cuda")
        for r in [(i + k // 2) % k for i in range(k)]:
            _lib.call("omg_forward_project", g.handle, r * n, n, ptr(img), ptr(y[r * n:]), None)
            _lib.call("omg_backward_project", g.handle, r * n, n, ptr(y[r * n:]), ptr(back), None, None)
        out.append((y.cpu().numpy(), back.cpu().numpy()))
        assert list_calls(g) == (0, 0 if gen else 2 * (k - 1))
    assert np.array_equal(out[0][0], out[1][0])
    assert rel_l2(out[0][1], out[1][1]) < BAR


def test_detectors_within_the_image(cuda):
    """LORs that start in the image are traced: their lengths are not the crossings' steps."""
    import torch
    fov = 50.0
    grid = G.Grid.from_fov(20, 20, 9, fov, fov, 22.5)
    x = G.ring_sinogram_xy(24, 20, 1.5, 20.0)
    z = np.random.default_rng(1).uniform(-10.0, 10.0, (40, 2)).astype(np.float32)
    n = 40 * 480
    img, y, meas = torch.rand(grid.N, device="cuda"), torch.rand(n, device="cuda"), torch.rand(n, device="cuda")
    geoms = [make_geom(grid, x, z, 24, 20, generic=gen) for gen in (False, True)]
    a, b = (_run(g, grid, 0, n, img, y, meas) for g in geoms)
    assert list_calls(geoms[0]) == (0, 0) and np.array_equal(a[0], b[0]) and rel_l2(a[1], b[1]) < BAR


def test_many_tiles(cuda):
    """More tiles than a workgroup counts in LDS."""
    import torch
    grid, x, z = _scanner(530, 530, 63, 24, 20, 33)
    n = 33 * 480
    img, y = torch.rand(grid.N, device="cuda"), torch.rand(n, device="cuda")
    out = []
    for gen in (False, True):
        geom = make_geom(grid, x, z, 24, 20, generic=gen)
        p, back = torch.empty(n, device="cuda"), torch.zeros(grid.N, device="cuda")
        _lib.call("omg_forward_project", geom.handle, 0, n, ptr(img), ptr(p), None)
        _lib.call("omg_backward_project", geom.handle, 0, n, ptr(y), ptr(back), None, None)
        out.append((p.cpu().numpy(), back.cpu().numpy()))
        assert list_calls(geom) == (0, 0 if gen else 2)
    assert np.array_equal(out[0][0], out[1][0])
    assert rel_l2(out[0][1], out[1][1]) < BAR


def test_several_passes(cuda):
    """140 planes of 224 x 224 bins: their records take two passes of plane groups, each with LORs off the lists. About
    1e5 terms per voxel, so the float atomics of the other kernels carry 2^-24 sqrt(1e5) = 2e-5; bar: four times that."""
    import torch
    grid, x, z = _scanner(20, 20, 9, 224, 224, 140)
    n = 140 * 224 * 224
    rng = np.random.default_rng(4)
    img = torch.from_numpy((rng.random(grid.N) + 0.5).astype(np.float32)).cuda()
    y, meas = torch.rand(n, device="cuda") - 0.3, torch.poisson(torch.full((n,), 2.0, device="cuda"))
    geoms = [make_geom(grid, x, z, 224, 224, generic=gen) for gen in (False, True)]
    a, b = (_run(g, grid, 0, n, img, y, meas) for g in geoms)
    assert list_calls(geoms[0]) == (0, 4)
    assert np.array_equal(a[0], b[0])
    e = [rel_l2(p, q) for p, q in zip(a[1:], b[1:])]
    print(f"[column] two passes rel-L2 {e}", flush=True)
    assert max(e) < 8e-5


def test_many_ranges_and_off(cuda):
    """An index table of 66 ranges keeps 64 lists and traces the others; reserved[3] and reserved[4] < 0 trace all."""
    import torch
    planes, per, k = 40, 66 * 7, 66
    grid, x, z = _scanner(20, 20, 9, 22, 21, planes)
    bins = np.random.default_rng(5).permutation(per).reshape(k, 7)
    index = (np.arange(planes)[None, :, None] * per + bins[:, None, :]).astype(np.uint32).ravel()
    img = torch.rand(grid.N, device="cuda") + 0.5
    n = planes * 7
    out = []
    for kw in ({}, {"generic": True}, {"x_fastest_only": True}, {"tube_budget_mib": -1}):
        g = make_geom(grid, x, z, 22, 21, meas_index=index, **kw)
        y = torch.empty(k * n, device="cuda")
        for s in range(k):
            _lib.call("omg_forward_project", g.handle, s * n, n, ptr(img), ptr(y[s * n:]), None)
        out.append(y.cpu().numpy())
        assert list_calls(g) == (0, 0 if kw else 64)
        assert np.array_equal(out[-1], out[0])


def test_not_finite(cuda):
    """A NaN or an infinity in the image or the data goes where the other kernels take it, and nowhere else."""
    import torch
    grid, x, z = _scanner(20, 20, 9, 24, 20, 40)
    n = 40 * 24 * 20
    rng = np.random.default_rng(2)
    img, y, meas = rng.random(grid.N) + 0.5, rng.random(n), rng.poisson(2.0, n)
    img[grid.N // 2 + 3], img[grid.N // 3], y[n // 2], y[n // 3] = np.inf, np.nan, np.nan, np.inf
    up = lambda a: torch.from_numpy(a.astype(np.float32)).cuda()
    a, b = (_run(make_geom(grid, x, z, 24, 20, generic=gen), grid, 0, n, up(img), up(y), up(meas))
            for gen in (False, True))
    assert np.array_equal(a[0], b[0], equal_nan=True)
    seen = b[4] > 0.5
    a[3], b[3] = a[3][seen], b[3][seen]
    for p, q in zip(a[1:], b[1:]):
        assert np.array_equal(np.isfinite(p), np.isfinite(q))
        ok = np.isfinite(q)
        assert rel_l2(p[ok], q[ok]) < BAR


@pytest.mark.parametrize("outlier", [2.0 ** 24, 2.0 ** 40, 1e30, 1e-30])
def test_range_of_values(cuda, outlier):
    """One LOR whose value is far from the others': the voxels beside it are as good as without it."""
    import torch
    grid, x, z = _scanner(33, 40, 15, 32, 30, 70)
    n = 70 * 960
    y = np.random.default_rng(6).random(n).astype(np.float32) + 0.5
    only = np.zeros(n, np.float32)
    only[37 * 960 + 15 * 32 + 14] = y[37 * 960 + 15 * 32 + 14] = outlier
    out = []
    for gen in (False, True):
        geom = make_geom(grid, x, z, 32, 30, generic=gen)
        back, path = torch.zeros(grid.N, device="cuda"), torch.zeros(grid.N, device="cuda")
        for v, to in ((y, back), (only, path)):
            _lib.call("omg_backward_project", geom.handle, 0, n, ptr(torch.from_numpy(v).cuda()), ptr(to), None, None)
        torch.cuda.synchronize()
        out.append((back.cpu().numpy(), path.cpu().numpy()))
        assert list_calls(geom) == (0, 0 if gen else 2)
    (a, pa), (b, pb) = out
    assert rel_l2(pa, pb) < BAR and np.count_nonzero(pb) > 20
    beside = pb == 0
    e = rel_l2(a[beside], b[beside]), rel_l2(a[~beside], b[~beside])
    print(f"[column] outlier {outlier:.1e}: rel-L2 {e}", flush=True)
    assert max(e) < BAR


@pytest.mark.parametrize("frames,planes", [(1, 40), (4, 64), (3, 97)])
def test_frames(cuda, frames, planes):
    """Two subset steps of a dynamic study, launched and replayed from a graph."""
    import torch
    grid, x, z = _scanner(21, 18, 11, 20, 16, planes)
    n, N = planes * 320, grid.N
    rng = np.random.default_rng(planes)
    up = lambda a: torch.from_numpy(a.astype(np.float32)).cuda()
    meas, x0 = up(rng.poisson(0.3, (frames, n))), up(rng.random((frames, N)) + 0.5)
    out = []
    for gen in (False, True):
        g = make_geom(grid, x, z, 20, 16, generic=gen)
        S, rhs, xs = torch.empty(N, device="cuda"), torch.zeros(frames, N, device="cuda"), x0.clone()
        y = torch.empty(frames, n, device="cuda")
        _lib.call("omg_frames_sensitivity", g.handle, 0, n, ptr(S), EPPS, None)
        tail = (0.0, 2.0, EPPS, 1, 128, 1, 0)
        for _ in range(2):
            _lib.call("omg_frames_osem_step", g.handle, 0, n, frames, ptr(xs), ptr(meas), n, ptr(S), ptr(rhs), None, *tail,
                      None)
        _lib.call("omg_frames_forward", g.handle, 0, n, frames, ptr(x0), ptr(y), n, None)
        torch.cuda.synchronize()
        res = [S.cpu().numpy(), xs.cpu().numpy(), y.cpu().numpy()]
        ints = [np.array([v], np.int64) for v in (0, n, 0)]
        h, xs = C.c_void_p(), x0.clone()
        torch.cuda.synchronize()
        _lib.call("omg_frames_graph_create", g.handle, 1, *(v.ctypes.data for v in ints), frames, ptr(xs), ptr(meas), n,
                  ptr(S), ptr(rhs), None, *tail, C.byref(h))
        for _ in range(2):
            _lib.call("omg_graph_launch", h, None)
            torch.cuda.synchronize()
            rhs.fill_(7.0)
        _lib.call("omg_graph_destroy", h)
        out.append(res + [xs.cpu().numpy()])
        assert list_calls(g) == (0, 0 if gen else 1 + 4 * frames)   # sensitivity, two steps, forward, captured step
    a, b = out
    assert np.array_equal(a[2], b[2])
    seen = b[0] > 0.5
    assert rel_l2(a[0], b[0]) < BAR
    for k in (1, 3):
        assert rel_l2(a[k][:, seen], b[1][:, seen]) < BAR


def test_first_call_beside_a_capture(cuda):
    """A handle's first projection, which builds its lists, while another thread captures: neither disturbs the other."""
    import threading
    import torch
    grid, x, z = _scanner(20, 20, 9, 24, 20, 40)
    n = 40 * 480
    img, out, want = torch.rand(grid.N, device="cuda"), torch.empty(n, device="cuda"), torch.empty(n, device="cuda")
    geom, gen = (make_geom(grid, x, z, 24, 20, generic=g) for g in (False, True))
    _lib.call("omg_forward_project", gen.handle, 0, n, ptr(img), ptr(want), None)
    side, a = torch.cuda.Stream(), torch.zeros(64, device="cuda")
    torch.cuda.synchronize()
    failed = []

    def project():
        try:
            torch.cuda.set_device(0)
            _lib.call("omg_forward_project", geom.handle, 0, n, ptr(img), ptr(out), C.c_void_p(side.cuda_stream))
        except Exception as e:
            failed.append(e)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        a.add_(1.0)
        t = threading.Thread(target=project)
        t.start()
        t.join()
        a.mul_(3.0)
    assert not failed
    for k in range(3):
        a.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float(a.sum()) == 64 * 3.0
    assert np.array_equal(out.cpu().numpy(), want.cpu().numpy())
    assert list_calls(geom) == (0, 1)


def _operands(grid, n, k):
    import torch
    return [torch.rand(grid.N, device="cuda") + 0.5 for _ in range(k)], [torch.empty(n, device="cuda") for _ in range(k)]


def test_projections_beside_each_other(cuda):
    """Forward projections of one handle on six streams and from six threads, with a backprojection between them."""
    import threading
    import torch
    grid, x, z = _scanner(64, 64, 31, 64, 60, 70)
    n = 70 * 64 * 60
    img, want = _operands(grid, n, 6)
    out = [torch.empty(n, device="cuda") for _ in img]
    y, back, ref = torch.rand(n, device="cuda"), torch.zeros(grid.N, device="cuda"), torch.zeros(grid.N, device="cuda")
    gen, geom = make_geom(grid, x, z, 64, 60, generic=True), make_geom(grid, x, z, 64, 60)
    for i, w in zip(img, want):
        _lib.call("omg_forward_project", gen.handle, 0, n, ptr(i), ptr(w), None)
    _lib.call("omg_backward_project", gen.handle, 0, n, ptr(y), ptr(ref), None, None)
    streams = [torch.cuda.Stream() for _ in img]
    torch.cuda.synchronize()

    def project(k):
        for _ in range(3):
            _lib.call("omg_forward_project", geom.handle, 0, n, ptr(img[k]), ptr(out[k]), C.c_void_p(streams[k].cuda_stream))

    for threads in (False, True):
        for o in out:
            o.zero_()
        back.zero_()
        torch.cuda.synchronize()
        ts = [threading.Thread(target=project, args=(k,)) for k in range(6)]
        for k, t in enumerate(ts):
            t.start() if threads else project(k)
            if k == 2:
                _lib.call("omg_backward_project", geom.handle, 0, n, ptr(y), ptr(back), None, None)
        for t in ts if threads else ():
            t.join()
        torch.cuda.synchronize()
        for o, w in zip(out, want):
            assert torch.equal(o, w)
        assert rel_l2(back.cpu().numpy(), ref.cpu().numpy()) < BAR


def test_captured_projection_outlives_the_buffers(cuda):
    """Projections captured on a handle with lists keep nothing of the handle's that later calls may grow and free."""
    import torch
    grid, x, z = _scanner(20, 20, 9, 24, 20, 70)
    n = 70 * 480
    (img,), (y,) = _operands(grid, n, 1)
    want = torch.empty(n, device="cuda")
    geom = make_geom(grid, x, z, 24, 20)
    side = torch.cuda.Stream()
    call = lambda out: _lib.call("omg_forward_project", geom.handle, 0, n, ptr(img), ptr(out),
                                 C.c_void_p(torch.cuda.current_stream().cuda_stream))
    call(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(y)
    back, S = torch.zeros(grid.N, device="cuda"), torch.zeros(grid.N, device="cuda")
    for k in range(3):
        _lib.call("omg_backward_project", geom.handle, 0, n, ptr(want), ptr(back), ptr(S), None)   # needs more memory
        img.mul_(1.5)
        y.zero_()
        graph.replay()
        call(want)
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    assert list_calls(geom) == (0, 7)     # the captured one traces


def test_frames_graph_takes_no_stack_it_does_not_use(cuda):
    """A graph whose steps go by columns holds no accumulator stack of image x frames."""
    import torch
    grid, x, z = _scanner(96, 96, 40, 20, 16, 40)
    frames, n, N = 128, 40 * 320, grid.N
    g = make_geom(grid, x, z, 20, 16)
    meas, xs = torch.ones(frames, n, device="cuda"), torch.ones(frames, N, device="cuda")
    S, rhs = torch.ones(N, device="cuda"), torch.zeros(frames, N, device="cuda")
    ints = [np.array([v], np.int64) for v in (0, n, 0)]
    tail = (0.0, 2.0, EPPS, 1, 128, 1, 0)
    _lib.call("omg_frames_osem_step", g.handle, 0, n, frames, ptr(xs), ptr(meas), n, ptr(S), ptr(rhs), None, *tail, None)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    h = C.c_void_p()
    _lib.call("omg_frames_graph_create", g.handle, 1, *(v.ctypes.data for v in ints), frames, ptr(xs), ptr(meas), n,
              ptr(S), ptr(rhs), None, *tail, C.byref(h))
    took = free - torch.cuda.mem_get_info()[0]
    _lib.call("omg_graph_destroy", h)
    print(f"[column] graph took {took >> 20} MiB beside a stack of {rhs.numel() * 4 >> 20} MiB", flush=True)
    assert list_calls(g) == (0, 2 * frames)
    assert took < rhs.numel() * 4
