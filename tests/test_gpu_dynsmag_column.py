"""The dynamic model on grids of one or few points a plane and as many planes
as its static scratch holds, against the oracle (1e-12 normwise relative).
The call only queues its two kernels: choosing the slabs of 2^21 planes takes
well under the 5 ms allowed for it (13 ms when every number of slabs was
tried)."""
import ctypes
import time

import numpy as np
import pytest
import torch

from conftest import normwise_rel
from emix3d_amd import _lib
from emix3d_amd.api import _ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1 << 21), (3, 2, 100003)])
def test_tall_columns(oracle, shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(nz)
    u, dvel = rng.standard_normal((3, nz, ny, nx)), rng.standard_normal((9, nz, ny, nx))
    jbn, delta = 0.5 + rng.random((11, nz, ny, nx)), 0.1 + rng.random((nz, ny, nx))
    gp = np.stack([jbn[4 * b] * dvel[3 * b + a] for a in range(3) for b in range(3)])
    ref = oracle.dynsmag(u, gp, delta)
    t = [torch.from_numpy(a).cuda() for a in (u, dvel, jbn, delta)]
    nut = torch.empty_like(t[3])
    args = (*shape, *map(_ptr, t), _ptr(nut), 0.0, None,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    host = []
    for _ in range(4):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        _lib.check("emx_dynsmag_noalloc", _lib.lib().emx_dynsmag_noalloc(*args))
        host.append(time.perf_counter() - t0)
    err = normwise_rel(nut.cpu().numpy(), ref)
    print(f"  {shape}: {err:.1e}, host {min(host) * 1e6:.0f} us", flush=True)
    assert err <= 1e-12
    assert min(host) < 5e-3
