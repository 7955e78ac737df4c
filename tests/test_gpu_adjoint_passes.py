"""The flux adjoint's passes (two that only solve and keep their results in the
output arrays, two that combine the three directions) and the gradient's
adjoint, on lines around the solve's chunk lengths (four points to a line of
256, eight above), with rows of lines that do not fill a workgroup and lines
all of whose points are edge rows, against the oracle; 1e-12 normwise."""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import Operator

pytestmark = pytest.mark.gpu
SID = {"c4": 0, "c6f": 1, "c6c": 2}


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def close(name, got, want):
    err = normwise_rel(got.cpu().numpy(), want)
    print(f"  {name}: {err:.1e}", flush=True)
    assert err <= 1e-12, name


@pytest.mark.parametrize("scheme", ["c4", "c6f", "c6c"])
@pytest.mark.parametrize("shape", [(5, 6, 7), (8, 9, 12), (256, 7, 13), (257, 17, 5), (9, 259, 6),
                                   (18, 6, 301), (512, 5, 9), (33, 31, 16)])
def test_flux_and_gradient_adj(oracle, scheme, shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(sum(shape))
    f = {k: rng.standard_normal((c, nz, ny, nx)) for k, c in
         (("rs", 5), ("rsv", 5), ("um", 5), ("u", 3), ("dvel", 9), ("db", 9), ("dt", 3))}
    vis = 1e-3 + rng.random((nz, ny, nx))
    jbn = 0.5 + rng.random((11, nz, ny, nx))
    ih = (nx - 1.0, ny - 1.0, nz - 1.0)
    op = Operator(nx, ny, nz, scheme)
    got = op.flujos_divergencia_all_adj(dev(f["rs"]), dev(f["rsv"]), dev(f["um"]), dev(f["u"]),
                                        dev(vis), dev(jbn), dev(f["dvel"]))
    ref = oracle.flux_div_all_adj(SID[scheme], f["rs"], f["rsv"], f["um"], f["u"], vis, jbn,
                                  f["dvel"], ih)
    for k in ("um_bar", "u_bar", "pres_bar", "vis_bar", "dvel_bar"):
        g, r = got[k].reshape(-1, nz, ny, nx), ref[k].reshape(-1, nz, ny, nx)
        for c in range(g.shape[0]):
            close(f"{k}[{c}]", g[c], r[c])
    ub, tb = op.deriv_vel_adj(dev(f["db"]), dev(f["dt"]))
    rub, rtb = oracle.deriv_vel_adj(SID[scheme], f["db"], f["dt"], ih)
    close("u_bar", ub, rub)
    close("temp_bar", tb, rtb)
