"""The number of paths a workgroup takes follows the length of the list (2, 4 or 8; lines at 512 and 1280 paths, FP64
512 and 1024): on both sides of each line the forward and the adjoint equal the calls with a fixed 8 (FP64: 4) or 1
paths per workgroup. Only the mapping of (path, energy) to lanes changes, so chi(k) is the same bit for bit; the
adjoint's FP64 sums over the energies are grouped the same way per path: 1e-12 of the largest component covers any
regrouping."""
import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
Q = np.arange(0.0, 18.0001, 0.05)


@pytest.mark.parametrize("npath", [1, 2, 511, 512, 513, 1024, 1025, 1279, 1280, 1281])
@pytest.mark.parametrize("case,npot,nleg", [("A018", 2, 2), ("A018", 2, 3), ("A014", 1, 2), ("A014", 1, 3)])
@pytest.mark.parametrize("prec", [32, 64])
def test_paths_per_workgroup_do_not_change_results(case, npot, nleg, npath, prec):
    from feffgpu_amd.paths import PathPlan
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = W.displaced(pos0, 0.07, 31)
    ipot = np.full(len(pos), npot)
    ipot[::4] = 1
    pl = W.concat([W.enumerate_paths(pos, a, ipot, 5.0, nleg, box=box, segment=i, nmax=nleg)
                   for i, a in enumerate(range(0, 64, 2))], nleg)
    sel = np.nonzero(pl.nleg == nleg)[0]
    sel = sel[np.arange(npath) % len(sel)]
    plan = PathPlan(str(GOLDEN / "validation" / case / "phase.pad"), Q, pl.atoms[sel], pl.nleg[sel], pl.absorber[sel],
                    pl.ipots[sel], pl.deg[sel], segment=np.zeros(npath, int), nseg=1, cell=float(box[0]),
                    precision=prec, device="cuda")
    p = torch.tensor(pos, device="cuda")
    g = torch.tensor(np.random.default_rng(5).normal(size=(1, len(Q))), device="cuda")
    out = []
    for gp in (0, 8 if prec == 32 else 4, 1):     # 8 FP64 paths do not fit one CU with their tables
        for kernel in (0, 1):
            for b in range(len(plan.buckets.kind)):
                plan.set_launch(kernel, b, gpaths=gp)
        chi = plan.forward(p)[0].clone()
        out.append((chi, plan.backward(p, g).clone()))
    for chi, grad in out[1:]:
        assert torch.equal(chi, out[0][0])
        assert float((grad - out[0][1]).abs().max()) <= 1e-12 * float(grad.abs().max())
