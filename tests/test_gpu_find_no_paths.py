"""The path finder where absorbers have no atom within reach: no path and the reference importance 1, whether a pass has
paths of other absorbers or none at all, with and without the degenerate merge."""
import numpy as np
import pytest
import torch

from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
PHASE = GOLDEN / "validation" / "A018" / "phase.pad"


@pytest.mark.parametrize("nlegmax", [2, 3, 4, 6])
@pytest.mark.parametrize("merge", [True, False])
def test_absorbers_without_neighbours(merge, nlegmax):
    from feffgpu_amd.pathfinder import GPUPathFinder
    fd = GPUPathFinder(str(PHASE), rmax=4.0, nlegmax=nlegmax, merge_degenerate=merge)
    lone = np.zeros((1, 3))
    apart = 20.0 * np.eye(3)
    for pos, ab in ((lone, [0]), (apart, [0]), (apart, [2, 0, 1, 1])):
        kept, ref = fd.enumerate_many(pos, None, ab, np.ones(len(pos), int))
        assert np.array_equal(ref, np.ones(len(ab), np.float32))
        for nleg, v in kept.items():
            assert all(t.shape[0] == 0 for t in v.values()) and v["coords"].shape == (0, nleg, 3)
    # one absorber with a neighbour among others without
    pair = np.concatenate([apart, apart[2:] + [0.0, 0.0, 2.5]])
    kept, ref = fd.enumerate_many(pair, None, [0, 2, 1], np.ones(4, int))
    assert kept[2]["slot"].tolist() == [1] and kept[2]["atoms"].tolist() == [[3]]
    assert ref[0] == ref[2] == 1.0 and ref[1] == float(kept[2]["xport"][0])
