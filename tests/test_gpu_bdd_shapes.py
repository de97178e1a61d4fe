"""The distance-driven kernels' variants at the sizes where they change, against the oracle (the same float
operations in the same order: 1e-6 relative L2, as the other distance-driven tests).

Odd volumes and panels (partial workgroups, column groups and z runs); more than 256 column groups; panel columns
much finer than a voxel (the backprojection's window does not hold them: taps from memory) and between (runs of 4);
a volume with more slices than LDS takes rows of.
"""
import numpy as np
import pytest

from omega_amd import geometry as G
from omega_amd.projector import projectorClass
from oracle import oracle as O
from tests.hip_helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,rows,cols,pitch,views,voxel", [
    ((33, 18, 21), 37, 29, 1.6, 7, 1.0),       # odd everything
    ((5, 7, 3), 3, 2, 4.0, 9, 2.0),            # less than one group, one wave
    ((20, 24, 30), 11, 2060, 0.05, 4, 1.0),    # 258 column groups; window passed
    ((112, 110, 111), 90, 200, 0.8, 3, 1.0),   # runs of 4
    ((130, 128, 131), 96, 88, 3.0, 2, 1.0),    # runs of 8, last one partial
    ((4, 5, 5003), 6, 40, 2.0, 2, 0.01),       # rows of more than 64 KB
    ((4, 5, 10301), 6, 40, 2.0, 2, 0.01),      # more slices than LDS rows
])
def test_shapes_match_oracle(cuda, shape, rows, cols, pitch, views, voxel):
    import torch
    grid = G.Grid.from_fov(*shape, *(n * voxel for n in shape))
    x, uv = G.cbct_tables(views, sod=240.0, sdd=400.0, pitch_u=pitch)
    p = projectorClass()
    p.CT = True
    p.projector_type = 5
    p.Nx, p.Ny, p.Nz = shape
    p.FOVa_x, p.FOVa_y, p.axial_fov = (n * voxel for n in shape)
    p.x, p.z = x.copy(), uv.copy()
    p.nRowsD, p.nColsD = rows, cols
    p.dPitchX = p.dPitchY = pitch
    p.addProjector()
    case = O.BDDCase(grid, rows, cols, x, uv, pitch, pitch)
    rng = np.random.default_rng(rows)
    vol = rng.random(grid.N).astype(np.float32)
    print(f"[bdd shapes] {shape} rows={rows} cols={cols}", flush=True)
    y = p.forwardProject(torch.as_tensor(vol, device=cuda), 0).cpu().numpy()
    w = rng.random(case.M).astype(np.float32)
    sens = torch.zeros(grid.N, device=cuda)
    b = p.backwardProject(torch.as_tensor(w, device=cuda), 0, sens=sens).cpu().numpy()
    b2 = p.backwardProject(torch.as_tensor(w, device=cuda), 0).cpu().numpy()
    yo = case.fp(vol)
    bo, so = case.bp(w, sens=True)
    e = [rel_l2(y, yo), rel_l2(b, bo), rel_l2(sens.cpu().numpy(), so), rel_l2(b2, bo)]
    print("  rel-L2 fp %.2e bp %.2e sens %.2e bp alone %.2e" % tuple(e), flush=True)
    assert max(e) < 1e-6
