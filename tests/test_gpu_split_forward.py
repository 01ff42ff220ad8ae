"""Long lists run the forward as three kernels (geometry records, amplitudes, fine grid; more than 1280 paths) through
the output's own rows: the same paths in short lists, which run as one kernel, give the same. FP64 1e-12 of the largest
value; FP32 2e-6 (the operations are the same; a last bit of the float32 results is all that could differ).
Also where the rows are too short for that (few q points, six legs into cchi) and where a path is invalid (NaN in its
rows only)."""
import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN, load_case

pytestmark = pytest.mark.gpu
TOL = {32: 2e-6, 64: 1e-12}


@pytest.mark.parametrize("nk", [3, 119, 120, 361])
@pytest.mark.parametrize("case,npot,nleg", [("A018", 2, 2), ("A018", 2, 3), ("A014", 1, 2), ("A014", 1, 3),
                                            ("A018", 2, 4)])
@pytest.mark.parametrize("prec", [32, 64])
def test_path_list(case, npot, nleg, nk, prec):
    from feffgpu_amd.paths import PathPlan
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = W.displaced(pos0, 0.07, 31)
    ipot = np.full(len(pos), npot)
    ipot[::4] = 1
    pl = W.concat([W.enumerate_paths(pos, a, ipot, 5.0, nleg, box=box, segment=i, nmax=nleg)
                   for i, a in enumerate(range(0, 64, 2))], nleg)
    sel = np.nonzero(pl.nleg == nleg)[0]
    sel = sel[np.arange(1301) % len(sel)]
    q = np.linspace(0.0, 17.9, nk)
    p = torch.tensor(pos, device="cuda")

    sigma2 = np.linspace(0, 0.01, len(sel))

    def chi(a, b, keep=False):
        r = sel[a:b]
        plan = PathPlan(str(GOLDEN / "validation" / case / "phase.pad"), q, pl.atoms[r], pl.nleg[r], pl.absorber[r],
                        pl.ipots[r], pl.deg[r], segment=np.arange(len(r)), nseg=len(r), sigma2=sigma2[a:b],
                        cell=float(box[0]), precision=prec, device="cuda")
        return plan.forward(p, keep=keep)[0].clone()

    long, kept = chi(0, 1301), chi(0, 1301, keep=True)
    short = torch.cat([chi(0, 700), chi(700, 1301)])
    assert torch.equal(long, kept)
    assert float((long - short).abs().max()) <= TOL[prec] * float(short.abs().max())


@pytest.mark.parametrize("case,nleg", [("L001", 3), ("L001", 5), ("L001", 6), ("A018", 3), ("A014", 3), ("A014", 2)])
@pytest.mark.parametrize("prec,dt", [(32, torch.complex64), (64, torch.complex128)])
def test_cchi(case, nleg, prec, dt):
    from feffgpu_amd.stage import GPUPathStage
    phase, paths, _, _ = load_case("validation/" + case)
    st = GPUPathStage(str(phase), dtype=dt)
    base = [x for x in paths if x.nleg == nleg][:4]
    rng = np.random.default_rng(nleg)
    c = np.stack([base[i % len(base)].coords for i in range(1285)])
    c[:, 1:] += rng.normal(0, 0.05, c[:, 1:].shape)
    ip = np.stack([base[i % len(base)].ipots for i in range(1285)]).astype(np.int64)
    bad = [0, 640, 1284]
    ip[bad, 1] = 99
    ct, it = torch.tensor(c, device="cuda"), torch.tensor(ip, device="cuda")
    long, reff = st._cchi_raw(ct, it)[:2]
    short = [st._cchi_raw(ct[a:a + 650].contiguous(), it[a:a + 650].contiguous())[:2] for a in (0, 650)]
    ok = torch.ones(1285, dtype=torch.bool, device="cuda")
    ok[bad] = False
    s = torch.cat([x[0] for x in short])
    assert bool(torch.view_as_real(long[~ok]).isnan().all()) and bool(torch.view_as_real(s[~ok]).isnan().all())
    d = (long[ok] - s[ok]).abs().amax(1)
    assert bool((d <= TOL[prec] * s[ok].abs().amax(1)).all())
    assert torch.equal(reff[ok], torch.cat([x[1] for x in short])[ok])
