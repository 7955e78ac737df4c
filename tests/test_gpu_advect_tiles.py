"""The level-set advection step on the GPU against the oracle where its tiles
(32 x 8 or 16 x 16 columns of the padded grid, slabs of 2 to 8 planes) end:
padded sides one below, at and one above a tile, the smallest grids (every
stencil reaches a ghost layer), slabs cut short.  The velocity takes both
signs and exact zeros in every component and the boxes of a batch differ in
tile shape; 1e-12 normwise relative, as the step's other comparisons."""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import Batch, Operator, fields

pytestmark = pytest.mark.gpu
SHAPES = [(5, 5, 5), (6, 38, 7), (21, 13, 9), (22, 14, 8), (23, 15, 7), (38, 22, 6), (54, 6, 6),
          (150, 142, 86)]


def problem(shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(sum(shape))
    f = fields.stage_fields(*shape, 63, curvilinear=True, turbulent=False)
    x = f["x"].numpy()
    phi = np.sqrt(((x - 0.45) ** 2).sum(0)) - 0.3 + 0.01 * np.sin(17.0 * x[0] + 11.0 * x[2])
    vel = rng.standard_normal((3, nz, ny, nx))
    vel[rng.random(vel.shape) < 0.1] = 0.0
    dxyz = (1.0 / (nx - 1), 1.0 / (ny - 1), 1.0 / (nz - 1))
    return np.ascontiguousarray(x), np.ascontiguousarray(phi), vel, dxyz, 0.02 * min(dxyz)


def close(name, got, want, before):
    err = normwise_rel(got.cpu().numpy(), want)
    print(f"  {name}: {err:.1e}", flush=True)
    assert err <= 1e-12, name
    assert normwise_rel(want, before) > 1e-8  # the step moved phi


@pytest.mark.parametrize("shape", SHAPES)
def test_advect_tiles_vs_oracle(oracle, shape):
    x, phi, vel, dxyz, dt = problem(shape)
    jbn = oracle.jacobeano(2, x)
    p = torch.from_numpy(phi.copy()).cuda()
    Operator(*shape, "c6c").advect_weno5(p, torch.from_numpy(vel).cuda(),
                                         torch.from_numpy(jbn).cuda(), dxyz, dt)
    close(f"phi {shape}", p, oracle.ls_advect_weno5(phi, vel, jbn, dxyz, dt), phi)


@pytest.mark.parametrize("count", [1, 7, 8])
def test_batched_advect_tiles_vs_oracle(oracle, count):
    shapes = SHAPES[:count]
    b = Batch(shapes, "c6c")
    want, phis = [], []
    for i, shape in enumerate(shapes):
        nx, ny, nz = shape
        x, phi, vel, dxyz, dt = problem(shape)
        jbn = oracle.jacobeano(2, x)
        p = torch.from_numpy(phi.copy()).cuda()
        b.bind(i, torch.from_numpy(vel).cuda(), torch.from_numpy(jbn).cuda(), p,
               torch.empty((9, nz, ny, nx), dtype=torch.float64, device="cuda"),
               torch.empty((nz, ny, nx), dtype=torch.float64, device="cuda"),
               (nx - 1.0, ny - 1.0, nz - 1.0), dxyz, dt)
        phis.append(p)
        want.append((oracle.ls_advect_weno5(phi, vel, jbn, dxyz, dt), phi))
    b.stage()
    for shape, p, (w, phi) in zip(shapes, phis, want):
        close(f"phi {shape}", p, w, phi)
