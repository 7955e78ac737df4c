"""The work area of the closure's training backward pass: one partial
gradient per workgroup, at most 256, for any number of rows; a call with just
that much writes nothing past it and gives the gradient it gives with more,
and one with a float less is refused."""
import ctypes

import pytest
import torch

from emix3d_amd import _lib
from emix3d_amd._lib import EmxError
from emix3d_amd.api import EMX_MLP_NPARAM, _fptr, mlp_backward_f32, mlp_forward_f32
from test_oracle_mlp import rand_norm, rand_params


def need(n):
    return int(_lib.lib().emx_mlp_backward_work(n))


@pytest.mark.parametrize("n,parts", [(1, 1), (64, 1), (65, 2), (16384, 256), (16385, 256),
                                     (65536, 256), (1 << 30, 256), ((1 << 31) - 1, 256)])
def test_work_is_the_partial_gradients(n, parts):
    assert need(n) == parts * EMX_MLP_NPARAM


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 64, 65, 1000, 16384, 20000])
def test_exact_work(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    P, norm = (torch.from_numpy(a).cuda() for a in (rand_params(31), rand_norm(32)))
    feat = torch.randn((n, 10), device="cuda", generator=g)
    dnu = torch.randn(n, device="cuda", generator=g)
    act, _ = mlp_forward_f32(P, norm, feat)
    pool = torch.full((need(n) + 4096,), float("nan"), device="cuda")
    ref, _ = mlp_backward_f32(P, norm, feat, act, dnu, torch.empty(2 * need(n), device="cuda"))
    grad, work = mlp_backward_f32(P, norm, feat, act, dnu, pool[:need(n)])
    assert work.numel() == need(n)
    assert torch.equal(grad, ref)
    assert torch.isnan(pool[need(n):]).all() and not torch.isnan(work).any()
    with pytest.raises(EmxError):
        _lib.call("emx_mlp_backward_f32", _fptr(P), _fptr(norm), _fptr(feat), _fptr(act), _fptr(dnu),
                  n, _fptr(grad), _fptr(work), need(n) - 1,
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
