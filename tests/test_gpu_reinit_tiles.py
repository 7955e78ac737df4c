"""Level-set reinitialisation on the GPU against the oracle where its tiles
(32 x 8 columns of the padded grid, slabs of 2 to 8 planes) end: padded
sides one below, at and one above a tile, slabs of the full height.  The
fields have ridges, valleys and exact zeros, where an axis needs neither, one
or both of its one-sided derivatives.  1e-12 normwise relative, as the
reinitialisation's other comparisons."""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import Operator, fields

pytestmark = pytest.mark.gpu


def kinked(x):
    """A union of two balls cut by a slab, zero on a block of points."""
    r = lambda c: np.sqrt(((x - np.array(c).reshape(3, 1, 1, 1)) ** 2).sum(0))  # noqa: E731
    d = np.minimum(r((0.3, 0.4, 0.5)) - 0.25, r((0.7, 0.6, 0.5)) - 0.2)
    d = np.maximum(d, np.abs(x[2] - 0.5) - 0.3) * (1.0 + 0.5 * x[0])
    d[2:4, 3:5, 1:6] = 0.0
    return np.ascontiguousarray(d)


@pytest.mark.parametrize("shape", [(21, 13, 9), (22, 14, 8), (23, 15, 7), (54, 6, 6),
                                   (150, 142, 86)])
def test_reinit_tiles_vs_oracle(oracle, shape):
    nx, ny, nz = shape
    f = fields.stage_fields(nx, ny, nz, 62, curvilinear=True, turbulent=False)
    x = np.ascontiguousarray(f["x"].numpy())
    jbn = oracle.jacobeano(2, x)
    phi = kinked(x)
    _, dmins, _ = oracle.inisgdm(x)
    dxyz = (1.0 / (nx - 1), 1.0 / (ny - 1), 1.0 / (nz - 1))
    deltamin = float(dmins.min())
    ref = oracle.ls_reinit(phi, jbn, dmins, dxyz, deltamin)
    op = Operator(*shape, "c6c")
    p = torch.from_numpy(phi.copy()).cuda()
    op.reinit_level_set(p, torch.from_numpy(jbn).cuda(), torch.from_numpy(dmins).cuda(), dxyz,
                        deltamin)
    torch.cuda.synchronize()
    err = normwise_rel(p.cpu().numpy(), ref)
    print(f"  reinit {shape}: {err:.1e}", flush=True)
    assert err <= 1e-12
