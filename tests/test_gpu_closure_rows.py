"""The closure's training passes at row counts around their tiles (16 and 32
rows per wavefront, 64 per workgroup, the last tile partly filled), against
the network in FP64.  Tolerances: FP32 sums of 64 terms over three layers
(forward, 1e-5) and of those over the rows (gradient, 1e-4), normwise."""
import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd.api import mlp_backward_f32, mlp_forward_f32
from test_oracle_mlp import rand_norm, rand_params

pytestmark = pytest.mark.gpu


def preactivations(P, norm, feat):
    """z1, z2, z3, z4 of every row, [n][193], in FP64."""
    P, norm = P.astype(np.float64), norm.astype(np.float64)
    h = (feat - norm[:10]) * norm[10:20]
    at, out = 0, []
    for fan_in, fan_out in ((10, 64), (64, 64), (64, 64), (64, 1)):
        W = P[at:at + fan_in * fan_out].reshape(fan_out, fan_in)
        at += fan_in * fan_out
        z = h @ W.T + P[at:at + fan_out]
        at += fan_out
        out.append(z)
        h = z / (1.0 + np.exp(-z))
    return np.concatenate(out, axis=1)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 63, 64, 65, 129, 1000, 16385])
def test_training_rows(oracle, n):
    P, norm = rand_params(31), rand_norm(32)
    rng = np.random.default_rng(n)
    feat = rng.standard_normal((n, 10)).astype(np.float32)
    dnu = rng.standard_normal(n).astype(np.float32)
    Pd, nd, fd = (torch.from_numpy(a).cuda() for a in (P, norm, feat))
    act, nu = mlp_forward_f32(Pd, nd, fd)
    ref = oracle.mlp_forward(P, norm, feat.astype(np.float64))
    assert normwise_rel(nu.cpu().numpy(), ref) <= 1e-5
    z = preactivations(P, norm, feat.astype(np.float64))
    assert normwise_rel(act.cpu().numpy(), z) <= 1e-5
    grad, _ = mlp_backward_f32(Pd, nd, fd, act, torch.from_numpy(dnu).cuda())
    gref = oracle.mlp_grad(P, norm, feat.astype(np.float64), dnu.astype(np.float64))
    assert normwise_rel(grad.cpu().numpy(), gref) <= 1e-4
