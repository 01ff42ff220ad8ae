"""A shallow copy of a plan shares its buffers and its side streams: they go back to the library's pool with the last of
the two, not while the copy still uses them."""
import copy
import gc

import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu


def _free_sets():
    """The two sets that were given back last; they are back in the pool (of at most 16) afterwards."""
    from feffgpu_amd import _native as N
    got = [N.lib().fm_overlap_acquire() for _ in range(2)]
    for s in got:
        N.lib().fm_overlap_release(s)
    return got


def test_a_copy_outlives_its_plan():
    from feffgpu_amd.paths import PathPlan
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = torch.tensor(W.displaced(pos0, 0.07, 3), device="cuda")
    pl = W.enumerate_paths(pos.cpu().numpy(), 0, np.full(len(pos0), 2), 4.6, 4, box=box, segment=0, nmax=4)
    plan = PathPlan(str(GOLDEN / "validation" / "A018" / "phase.pad"), np.arange(0.0, 18.0001, 0.05), pl.atoms, pl.nleg,
                    pl.absorber, pl.ipots, pl.deg, cell=float(box[0]))
    want = plan.forward(pos)[0].clone()
    other = copy.copy(plan)
    mine = other._overlap
    assert mine
    del plan
    gc.collect()
    torch.cuda.synchronize()
    assert mine not in _free_sets()
    assert torch.equal(other.forward(pos)[0], want)
    torch.cuda.synchronize()
    del other
    gc.collect()
    assert mine in _free_sets()
