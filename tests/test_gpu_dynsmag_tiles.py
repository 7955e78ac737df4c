"""The dynamic Smagorinsky model on the GPU against the oracle where its tiles
(30 x 14 columns, slabs of any height) end: sides one below, at and one above
a tile, single slabs and cut ones, and the outputs placed over an input the
second pass does not read at other points.  1e-12 normwise relative."""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import Operator

pytestmark = pytest.mark.gpu


def problem(shape, oracle):
    nx, ny, nz = shape
    rng = np.random.default_rng(sum(shape))
    f = {"u": rng.standard_normal((3, nz, ny, nx)), "dvel": rng.standard_normal((9, nz, ny, nx)),
         "jbn": 0.5 + rng.random((11, nz, ny, nx)), "delta": 0.1 + rng.random((nz, ny, nx))}
    gp = np.stack([f["jbn"][4 * b] * f["dvel"][3 * b + a] for a in range(3) for b in range(3)])
    return f, oracle.dynsmag(f["u"], np.ascontiguousarray(gp), f["delta"])


def dev(a):
    return torch.from_numpy(a.copy()).cuda()


def close(name, got, want):
    err = normwise_rel(got.cpu().numpy(), want)
    print(f"  {name}: {err:.1e}", flush=True)
    assert err <= 1e-12, name


@pytest.mark.parametrize("shape", [(5, 5, 5), (29, 13, 6), (30, 14, 7), (31, 15, 8), (61, 29, 40),
                                   (20, 200, 33), (150, 9, 70)])
def test_dynsmag_tiles_vs_oracle(oracle, shape):
    f, ref = problem(shape, oracle)
    assert (ref > 0).any() and (ref == 0).any()
    op = Operator(*shape, "c6c")
    u, dvel, jbn, delta = (dev(f[k]) for k in ("u", "dvel", "jbn", "delta"))
    nut, vis = torch.empty_like(delta), torch.empty_like(delta)
    op.dynsmag(u, dvel, jbn, delta, nut=nut, c4=1e-3, vis=vis)
    close(f"nut {shape}", nut, ref)
    close(f"vis {shape}", vis, 1e-3 + ref)


@pytest.mark.parametrize("over", ["u", "dvel", "jbn", "delta"])
def test_dynsmag_output_over_an_input(oracle, over):
    shape = (47, 33, 21)
    f, ref = problem(shape, oracle)
    op = Operator(*shape, "c6c")
    t = {k: dev(f[k]) for k in f}
    nut = t[over][0] if t[over].ndim == 4 else t[over]
    op.dynsmag(t["u"], t["dvel"], t["jbn"], t["delta"], nut=nut)
    close(f"nut over {over}", nut, ref)
