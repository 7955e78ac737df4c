"""Line passes of more than 1024 workgroups, whose line groups are dealt to
the XCDs in runs: the gradient, the gradient fused with the divergence and
the flux divergence, with plans of 8, 16, 32 and 64 lines and group counts
that are a multiple of 128, of 8 and of neither, and the same grids with
fewer workgroups; against the oracle, 1e-12 normwise relative."""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import Operator, fields

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def close(name, got, want):
    err = normwise_rel(got.cpu().numpy(), want)
    print(f"  {name}: {err:.1e}", flush=True)
    assert err <= 1e-12, name


def workgroups(shape, d, lines, parts):
    nx, ny, nz = shape
    return -(-nx // lines) * (nz if d == 1 else ny) * parts


# kind and chunk, lines per workgroup
PLANS = [(1, 8, 64), (2, 4, 32), (3, 8, 16), (4, 4, 8)]


@pytest.mark.parametrize("shape,plan,above", [
    ((64, 80, 80), 3, True),   # 640 groups a part: 5 * 128
    ((61, 77, 93), 3, True),
    ((128, 83, 80), 2, True),
    ((130, 79, 64), 2, True),
    ((400, 45, 41), 1, True),
    ((700, 48, 47), 0, True),
    ((37, 41, 33), 3, False), ((37, 41, 33), 2, False), ((65, 23, 24), 1, False),
    ((140, 23, 24), 0, False)])
def test_runs(oracle, shape, plan, above):
    kind, chunk, lines = PLANS[plan]
    for d in (1, 2):  # the gradient's fields run as two parts, the fluxes as four
        assert workgroups(shape, d, lines, 2) > 1024 if above else workgroups(shape, d, lines, 4) <= 1024
    f = fields.stage_fields(*shape, 73, curvilinear=True, turbulent=True)
    z = {k: np.ascontiguousarray(v.numpy()) for k, v in f.items()}
    jbn = oracle.jacobeano(2, z["x"])
    op = Operator(*shape, "c6c")
    for d in (1, 2):
        op.set_plan(d, kind, chunk)
    ih = op.default_ih()
    rdv, rdt = oracle.deriv_vel(2, z["u"], z["temp"], ih)
    dv, dt = op.deriv_vel(dev(z["u"]), dev(z["temp"]))
    close("dvel", dv, rdv)
    close("dtemp", dt, rdt)
    dv, div = op.grad_div(dev(z["u"]), jbn=dev(jbn))
    rdiv, _ = oracle.divergencia(2, np.concatenate([z["u"], np.zeros_like(z["u"])]), jbn, ih)
    close("dvel (grad_div)", dv, rdv)
    close("div", div, rdiv)
    vis = np.ascontiguousarray(1e-3 + 1e-3 * np.abs(z["u"][0]))
    rs, rsv = op.flujos_divergencia_all(dev(z["um"]), dev(z["u"]), dev(z["pres"]), dev(vis),
                                        dev(jbn), dev(rdv))
    for neq in range(1, 6):
        flux = oracle.flujos(neq, z["um"], z["u"], z["pres"], vis, jbn, rdv)
        rrs, rrsv = oracle.divergencia(2, flux, jbn, ih)
        close(f"rs{neq}", rs[neq - 1], rrs)
        close(f"rsv{neq}", rsv[neq - 1], rrsv)
