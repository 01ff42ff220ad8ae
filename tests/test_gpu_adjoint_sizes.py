"""The multiple-scattering adjoint at the edges of its launches: groups of 16 paths, four paths per workgroup of the
chain, 4, 8 or 16 (path, scatterer) units per workgroup of the streams (by the size of the launch), a partial last
group.

A path's gradient does not depend on the list it is in: rows of a call on many paths equal calls on one path. The
per-energy values are the same operations; only the FP64 sums over the energies are split differently (E <= 60 terms,
each within a few ulp of 1.1e-16), so 1e-11 of the path's largest component holds for both precisions. The FP32
gradient against the FP64 one: 1e-4 of the largest component, the bar of the finite-difference tests.
"""
import numpy as np
import pytest
import torch

from fixtures import load_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npath", [1, 3, 15, 16, 17, 33, 4111])
@pytest.mark.parametrize("case,nleg", [("validation/A018", 3), ("validation/L001", 4), ("validation/L001", 5),
                                       ("validation/L001", 6), ("validation/A014", 3), ("validation/A014", 4)])
def test_rows_equal_single_paths(case, nleg, npath):
    from feffgpu_amd.stage import GPUPathStage
    phase, paths, _, _ = load_case(case)
    base = [p for p in paths if p.nleg == nleg][:4]
    rng = np.random.default_rng(100 * nleg + npath)
    coords = np.stack([base[i % len(base)].coords for i in range(npath)])
    coords[:, 1:] += rng.normal(0, 0.08, coords[:, 1:].shape)
    ipots = np.stack([base[i % len(base)].ipots for i in range(npath)])
    pick = sorted({0, npath // 2, npath - 1, max(npath - 2, 0)})
    grads = {}
    for prec, dt in ((64, torch.complex128), (32, torch.complex64)):
        st = GPUPathStage(str(phase), dtype=dt)
        w = torch.tensor((np.random.default_rng(7).normal(size=(npath, st.E, 2)) @ [1, 1j]) *
                         np.exp(-0.1 * np.arange(st.E)), device="cuda", dtype=dt)
        wr = torch.linspace(-1, 1, npath, device="cuda", dtype=torch.float64)
        ct, it = torch.tensor(coords, device="cuda"), torch.tensor(ipots, device="cuda")
        grads[prec] = st._cchi_backward_raw(ct, it, w, wr)
        for i in pick:
            one = st._cchi_backward_raw(ct[i:i + 1].contiguous(), it[i:i + 1].contiguous(), w[i:i + 1].contiguous(),
                                        wr[i:i + 1].contiguous())[0]
            assert float((grads[prec][i] - one).abs().max()) <= 1e-11 * float(one.abs().max()), (prec, i)
    scale = grads[64].abs().amax(dim=(1, 2))
    assert bool(((grads[32] - grads[64]).abs().amax(dim=(1, 2)) <= 1e-4 * scale).all())
