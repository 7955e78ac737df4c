"""The compact filter's line passes against the oracle, 1e-12 normwise
relative per field: xi lines at the ends of each chunk length (one to four
points per lane in one launch, eight and sixteen field by field), and eta and
zeta passes of more than 1024 workgroups, whose line groups are dealt in
runs, five fields side by side, with group counts that are no multiple of 8
or 128 (a group left out or filtered twice shows)."""
import numpy as np
import pytest

from conftest import normwise_rel
from emix3d_amd import Operator
from test_gpu_filter import case, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,itf", [
    ((64, 9, 12), 1), ((65, 9, 12), 2), ((128, 9, 12), 1), ((129, 11, 12), 1), ((161, 9, 12), 3),
    ((192, 70, 60), 1), ((193, 9, 12), 1), ((260, 9, 12), 2), ((512, 9, 12), 1), ((520, 12, 9), 1),
    ((1024, 9, 8), 6), ((150, 50, 60), 4), ((133, 72, 61), 5)])
@pytest.mark.parametrize("cfilt", [0.49, 0.0])
def test_filter_lines(oracle, shape, itf, cfilt):
    um1, jbn = case(shape, sum(shape), oracle)
    ref, _, _, _ = oracle.filtrado(itf, um1, jbn, cfilt, 0.3)
    d = dev(um1)
    Operator(*shape, "c6c").filtrado(itf, d, dev(jbn), cfilt, 0.3)
    got = host(d)
    for m in range(5):
        err = normwise_rel(got[m], ref[m])
        print(f"  filter {shape} itf {itf} field {m}: {err:.1e}", flush=True)
        assert err <= 1e-12
