"""Values at and beyond the ends of the double range.

  * An infinity or NaN at one point of a xi line reaches every point of that
    line's derivatives, as the line's solve couples them all, and no other
    line, for every chunk length of the wavefront kind, alone and batched;
  * the level set's reinitialisation where phi0^2 + dmin^2 overflows (a
    spacing that freezes its points, a level set far from any interface)
    against the oracle, 1e-12 normwise relative;
  * an infinite feature of the closure's training pass gives infinities of
    the weights' signs in its row's first layer, and leaves the other rows.
"""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import Batch, Operator, fields
from emix3d_amd.api import mlp_forward_f32
from test_oracle_mlp import rand_norm, rand_params

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def two_phase(oracle, shape):
    """Metrics, a distorted distance, spacings and their least of a tanh grid."""
    x = np.ascontiguousarray(
        fields.stage_fields(*shape, 63, curvilinear=True, turbulent=False)["x"].numpy())
    d = np.sqrt(((x - 0.5) ** 2).sum(0)) - 0.3
    return oracle.jacobeano(2, x), np.ascontiguousarray(d * (1.0 + 2.0 * d)), oracle.inisgdm(x)[1]


def assert_line_only(got, clean, line):
    """Every value of the line (j, k) non-finite, the others as in clean."""
    bad = ~np.isfinite(got)
    assert bad[line].all()
    bad[line] = False
    assert not bad.any()
    got, clean = got.copy(), clean.copy()
    got[line] = clean[line] = 0.0
    assert np.array_equal(got, clean)


# one, two, four, eight and sixteen points to a lane; a few lines past and
# many past what one wavefront takes at a time
@pytest.mark.parametrize("scheme", ["c4", "c6f", "c6c"])
@pytest.mark.parametrize("shape", [(60, 9, 8), (128, 9, 8), (140, 9, 8), (256, 70, 64),
                                   (300, 9, 8), (700, 9, 8)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_nonfinite_xi_line(scheme, shape, value):
    nx, ny, nz = shape
    op = Operator(*shape, scheme)
    rng = np.random.default_rng(nx)
    f = rng.standard_normal((4, nz, ny, nx))
    clean = [op.derivative(dev(f[0]), 0), *op.deriv_vel(dev(f[:3]), dev(f[3]))]
    clean = [t.cpu().numpy() for t in clean]
    line = (5, 7)
    f[0][line][nx // 3] = value
    got = op.derivative(dev(f[0]), 0).cpu().numpy()
    assert_line_only(got, clean[0], line)
    dvel, dtemp = (t.cpu().numpy() for t in op.deriv_vel(dev(f[:3]), dev(f[3])))
    assert_line_only(dvel[0], clean[1][0], line)  # du/dxi
    assert np.array_equal(dvel[1:3], clean[1][1:3])  # the fields solved beside u
    assert np.array_equal(dtemp, clean[2])


def test_nonfinite_xi_line_batched():
    dims = [(60, 9, 8), (128, 9, 8), (140, 9, 8), (200, 9, 8), (300, 9, 8)]
    out = []
    for value in (0.25, np.nan):
        b, keep = Batch(dims, "c6c"), []
        for i, d in enumerate(dims):
            z = fields.batch_box(d, 7 + i, device="cuda")
            z["u"][1, 5, 7, d[0] // 3] = value
            z["jbn"] = Operator(*d, "c6c").jacobeano(z["x"])
            dvel, div = (torch.empty(s + d[::-1], dtype=torch.float64, device="cuda")
                         for s in ((9,), ()))
            b.bind(i, z["u"], z["jbn"], z["phi"], dvel, div, z["ih"], z["dxyz"], z["dt"])
            keep.append((z, dvel, div))
        b.stage()
        torch.cuda.synchronize()
        out.append([k[1][1].cpu().numpy() for k in keep])  # dv/dxi
    for clean, got in zip(*out):
        assert_line_only(got, clean, (5, 7))


@pytest.mark.parametrize("value", [1e160, 1e200, -1e200, np.inf])
def test_reinit_frozen_points(oracle, value):
    """An infinite or overflowing dmin freezes its points: sign(phi) is 0."""
    shape = (30, 20, 25)
    jbn, phi, dmins = two_phase(oracle, shape)
    deltamin = float(dmins.min())
    frozen = np.zeros(phi.shape, bool)
    frozen[5:9, 4:15, 10:20] = True
    dmins = np.where(frozen, value, dmins)
    dxyz = tuple(1.0 / (n - 1) for n in shape)
    ref = oracle.ls_reinit(phi, jbn, dmins, dxyz, deltamin)
    p = dev(phi)
    Operator(*shape, "c6c").reinit_level_set(p, dev(jbn), dev(dmins), dxyz, deltamin)
    got = p.cpu().numpy()
    # thirty stages that re-round phi
    assert normwise_rel(ref[frozen], phi[frozen]) <= 7e-15
    assert normwise_rel(got[frozen], phi[frozen]) <= 7e-15
    assert normwise_rel(got, ref) <= 1e-12


@pytest.mark.parametrize("value", [1e160, -1e200])
def test_reinit_far_from_any_interface(oracle, value):
    shape = (17, 12, 9)
    jbn, phi, dmins = two_phase(oracle, shape)
    phi = np.full_like(phi, value)
    dxyz = tuple(1.0 / (n - 1) for n in shape)
    p = dev(phi)
    Operator(*shape, "c6c").reinit_level_set(p, dev(jbn), dev(dmins), dxyz, float(dmins.min()))
    ref = oracle.ls_reinit(phi, jbn, dmins, dxyz, float(dmins.min()))
    assert normwise_rel(ref / value, np.ones_like(phi)) <= 7e-15
    assert normwise_rel(p.cpu().numpy() / value, np.ones_like(phi)) <= 7e-15


@pytest.mark.parametrize("value", [np.inf, -np.inf])
@pytest.mark.parametrize("feature", [0, 1, 9])
def test_infinite_feature(feature, value):
    P, norm = rand_params(31), rand_norm(32)
    feat = np.random.default_rng(feature).standard_normal((50, 10)).astype(np.float32)
    clean, _ = mlp_forward_f32(dev(P), dev(norm), dev(feat))
    feat[33, feature] = value
    act, _ = mlp_forward_f32(dev(P), dev(norm), dev(feat))
    act, clean = act.cpu().numpy(), clean.cpu().numpy()
    w = P[:640].reshape(64, 10)[:, feature] * norm[10 + feature]
    assert np.array_equal(act[33, :64], np.copysign(np.float32(np.inf), w * value))
    assert np.array_equal(np.delete(act, 33, 0), np.delete(clean, 33, 0))
