"""The transposed solve of one, two, three and four fields (the derivative's,
the divergence's and the gradient's adjoints) against the oracle, 1e-12
normwise: lines of up to 256 points (chunks of four) and of 257 to 512
(chunks of eight), these with fewer and with more than 64 workgroups of
sixteen lines, below and above 1024 workgroups (dealt in runs), with rows
that end inside a group of eight or sixteen lines."""
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


@pytest.mark.parametrize("scheme,shape", [
    ("c4", (33, 16, 500)), ("c6f", (19, 300, 9)), ("c6c", (300, 7, 11)), ("c6c", (512, 6, 7)),
    ("c6c", (40, 257, 24)), ("c4", (37, 512, 30)), ("c6f", (70, 24, 401)), ("c6c", (265, 270, 70)),
    ("c6f", (130, 131, 64)), ("c6c", (17, 9, 256))])
def test_adjoints_by_line_length(oracle, scheme, shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(sum(shape))
    db = rng.standard_normal((9, nz, ny, nx))
    dt = rng.standard_normal((3, nz, ny, nx))
    jbn = 0.5 + rng.random((11, nz, ny, nx))
    ih = (nx - 1.0, ny - 1.0, nz - 1.0)
    sid = SID[scheme]
    op = Operator(*shape, scheme)
    for d in range(3):
        close(f"derivative {d}", op.derivative_adj(dev(db[d]), d),
              oracle.deriv3d_adj(sid, d, db[d], ih[d]))
    fb = op.divergencia_adj(dev(db[0]), dev(db[1]), dev(jbn))
    ref = oracle.divergencia_adj(sid, np.ascontiguousarray(db[0]), np.ascontiguousarray(db[1]), jbn, ih)
    for c in range(6):
        close(f"flux {c}", fb[c], ref[c])
    ref, rt = oracle.deriv_vel_adj(sid, db, dt, ih)
    ub, tb = op.deriv_vel_adj(dev(db), dev(dt))
    close("u", ub, ref)
    close("temperature", tb, rt)
    ub, tb = op.deriv_vel_adj(dev(db))
    assert tb is None
    close("u alone", ub, ref)
