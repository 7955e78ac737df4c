"""The batched wavefront kind along x, whose kernel is that of the longest
chunk any box needs (1, 2, 3, 4 or 8 points per lane): longest lines at and
around each chunk length's limit, every scheme, beside boxes of shorter
chunks, against the oracle (1e-12 normwise relative); and the autotuner,
which times it once."""
import pytest

from test_gpu_batch import check, make_batch, reference, reset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,sid", [("c4", 0), ("c6f", 1), ("c6c", 2)])
@pytest.mark.parametrize("longest", [64, 65, 128, 129, 192, 193, 256, 257, 512])
def test_longest_chunk(oracle, scheme, sid, longest):
    dims = [(20, 8, 7), (longest, 9, 8), (max(longest // 2, 9), 7, 9), (longest, 6, 5)]
    b, boxes = make_batch(dims, scheme)
    refs = [reference(oracle, z, sid) for z in boxes]
    assert b.get_plan(0)[0] == 0
    for graph in (False, True):
        reset(boxes)
        b.stage(graph=graph)
        check(oracle, boxes, refs, f"{scheme} {longest} graph={graph}")


def test_tuner_times_the_wave_kind_once(oracle):
    """All wavefront shapes that fit are one kernel: the shortest is the one
    that is kept, if any."""
    b, boxes = make_batch([(130, 90, 60), (190, 70, 50), (33, 80, 60)])
    for _ in range(3):
        b.tune(reps=3)
        lg, c = b.get_plan(0)
        assert lg != 0 or c == 4
    refs = [reference(oracle, z) for z in boxes]
    reset(boxes)
    b.stage()
    check(oracle, boxes, refs, "tuned")
