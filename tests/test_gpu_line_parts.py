"""The gradient's and the flux divergence's line passes, which solve their
fields as parts of one launch on the strided kinds and launch by launch on
the wavefront kind, and the slab rule of sgdm's plane march, against the
oracle; 1e-12 normwise relative, sgdm's switch decisions equal."""
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


# line groups of a direction a multiple of 128, of 8 and of neither; more
# than one group along a row and a last one that is not full
@pytest.mark.parametrize("plan", [(0, 1), (1, 8), (2, 4), (2, 16), (3, 8), (4, 4)])
@pytest.mark.parametrize("shape", [(37, 61, 43), (64, 32, 32), (65, 19, 24)])
def test_stage_parts(oracle, plan, shape):
    f = fields.stage_fields(*shape, 71, curvilinear=True, turbulent=True)
    z = {k: np.ascontiguousarray(v.numpy()) for k, v in f.items()}
    jbn = oracle.jacobeano(2, z["x"])
    op = Operator(*shape, "c6c")
    for d in (1, 2):
        op.set_plan(d, *plan)
    ih = op.default_ih()
    rdv, rdt = oracle.deriv_vel(2, z["u"], z["temp"], ih)
    dv, dt = op.deriv_vel(dev(z["u"]), dev(z["temp"]))
    close("dvel", dv, rdv)
    close("dtemp", dt, rdt)
    vis = np.ascontiguousarray(1e-3 + 1e-3 * np.abs(z["u"][0]))
    rs, rsv = op.flujos_divergencia_all(dev(z["um"]), dev(z["u"]), dev(z["pres"]), dev(vis),
                                        dev(jbn), dev(rdv))
    for neq in range(1, 6):
        flux = oracle.flujos(neq, z["um"], z["u"], z["pres"], vis, jbn, rdv)
        rrs, rrsv = oracle.divergencia(2, flux, jbn, ih)
        close(f"rs{neq}", rs[neq - 1], rrs)
        close(f"rsv{neq}", rsv[neq - 1], rrsv)


# slabs of 16, 8, 4 and 2 planes, the last one cut short
@pytest.mark.parametrize("shape", [(512, 512, 17), (512, 505, 9), (512, 250, 15), (33, 9, 5)])
def test_sgdm_slabs(oracle, shape):
    f = fields.stage_fields(*shape, 72, curvilinear=True, turbulent=False)
    z = {k: np.ascontiguousarray(f[k].numpy()) for k in ("x", "u")}
    jbn = oracle.jacobeano(2, z["x"])
    sgd, _, _ = oracle.inisgdm(z["x"])
    op = Operator(*shape, "c6c")
    dv, _ = op.deriv_vel(dev(z["u"]))
    amut, vis, _ = op.viscosidad_t(dev(z["u"]), dv, dev(jbn), dev(sgd), 1e-3)
    ra, rv, _ = oracle.sgdm(z["u"], dv.cpu().numpy(), jbn, sgd, 1e-3)
    close("amut", amut, ra)
    close("vis", vis, rv)
    assert np.array_equal(amut.cpu().numpy() == 0.0, ra == 0.0)
