"""The ordered segment sum on both sides of its rule (16 or 64 k-points per workgroup by the number of segments) and at
the edges of its tiles, against the sum of the plan's own chi_path in numpy: FP64 sums of at most 400 terms, 1e-13 of the
sum of the absolute values."""
import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nseg", [1, 3, 42, 43, 300])
@pytest.mark.parametrize("nk", [1, 15, 16, 17, 64, 65, 361])
@pytest.mark.parametrize("prec", [32, 64])
def test_segment_sum(nseg, nk, prec):
    from feffgpu_amd.paths import PathPlan
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = W.displaced(pos0, 0.07, 31)
    pl = W.concat([W.enumerate_paths(pos, a, np.full(len(pos), 2), 4.4, 3, box=box, segment=0, nmax=3)
                   for a in range(0, 20)], 3)
    pick = np.arange(400) % len(pl.nleg)
    seg = np.random.default_rng(nseg).integers(0, nseg, 400)       # some segments have no path
    q = np.linspace(0.0, 17.9, nk)
    plan = PathPlan(str(GOLDEN / "validation" / "A018" / "phase.pad"), q, pl.atoms[pick], pl.nleg[pick],
                    pl.absorber[pick], pl.ipots[pick], pl.deg[pick], segment=seg, nseg=nseg, cell=float(box[0]),
                    precision=prec, device="cuda")
    chi_seg, chi_path, _ = plan.forward(torch.tensor(pos, device="cuda"))
    terms = chi_path.double().cpu().numpy() * pl.deg[pick][:, None]
    want, scale = np.zeros((nseg, nk)), np.zeros((nseg, nk))
    np.add.at(want, seg, terms)
    np.add.at(scale, seg, np.abs(terms))
    assert (np.abs(chi_seg.cpu().numpy() - want) <= 1e-13 * scale + 1e-300).all()
