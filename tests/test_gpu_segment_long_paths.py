"""The segment sum on both sides of its rule for a list with buckets of 2 to 8 legs: FP64 sums of the plan's own chi_path,
1e-13 of the sum of the absolute values."""
import numpy as np
import pytest
import torch

from feffgpu_amd.feffio import read_paths_dat
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nseg", [1, 42, 43])
@pytest.mark.parametrize("prec", [32, 64])
def test_two_to_eight_legs(nseg, prec):
    from feffgpu_amd.paths import PathPlan
    d = GOLDEN / "validation" / "L001"
    paths = read_paths_dat(d / "paths.dat")
    nmax = max(p.nleg for p in paths)
    pos, atoms = [np.zeros(3)], []
    for x in paths:
        atoms.append(list(range(len(pos), len(pos) + x.nleg - 1)) + [0] * (nmax - x.nleg))
        pos += list(x.coords[1:])
    deg = np.array([x.deg for x in paths], float)
    seg = np.random.default_rng(nseg).integers(0, nseg, len(paths))
    plan = PathPlan(str(d / "phase.pad"), np.arange(0.0, 18.0001, 0.05), np.array(atoms),
                    np.array([x.nleg for x in paths]), np.zeros(len(paths), int),
                    np.array([list(x.ipots) + [0] * (nmax - x.nleg) for x in paths]), deg, segment=seg, nseg=nseg,
                    precision=prec)
    assert nmax >= 7
    chi_seg, chi_path, _ = plan.forward(torch.tensor(np.array(pos), device="cuda"))
    terms = chi_path.double().cpu().numpy() * deg[:, None]
    want, scale = np.zeros(chi_seg.shape), np.zeros(chi_seg.shape)
    np.add.at(want, seg, terms)
    np.add.at(scale, seg, np.abs(terms))
    assert (np.abs(chi_seg.cpu().numpy() - want) <= 1e-13 * scale + 1e-300).all()
