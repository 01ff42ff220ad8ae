"""chi_fine with a dense interpolation matrix at the edges of its kernel's tiles: 64 paths and 32 q-points per workgroup,
4 rows of S per wavefront, 64 energies at a time (W's phase grid has more), against the formula in numpy.

Tolerances as for the larch convention: FP64 1e-10 (phases of a few hundred radians, 3e-14 each, E terms), FP32 2e-5
(float32 amplitude and angle, 2^-24 relative each, on phases below pi before the unwrap)."""
import numpy as np
import pytest
import torch

from fixtures import GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npath", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("nk", [1, 7, 8, 9, 64, 65, 361])
@pytest.mark.parametrize("phase", ["validation/A014", "W"])
@pytest.mark.parametrize("dtype,tol", [(torch.complex128, 1e-10), (torch.complex64, 2e-5)], ids=["fp64", "fp32"])
def test_dense_interpolation_edges(phase, dtype, tol, nk, npath):
    from feffgpu_amd.stage import GPUPathStage
    st = GPUPathStage(str(GOLDEN / phase / "phase.pad"), dtype=dtype)
    E = st.E
    rng = np.random.default_rng(npath * 1000 + nk)
    x = np.linspace(0.0, 1.0, E)
    # smooth amplitudes and phases that wrap several times (steps well below pi)
    a = 0.5 + rng.random((npath, 1)) + 0.3 * np.sin(7 * x * rng.random((npath, 1)))
    ph = rng.normal(size=(npath, 1)) + x * 25.0 * rng.uniform(-1, 1, (npath, 1))
    cc = a * np.exp(1j * ph)
    reff = rng.uniform(2.0, 6.0, npath)
    q = np.linspace(0.0, 18.0, nk)
    S = rng.random((nk, E)) / E
    got = st.chi_fine(torch.tensor(cc, device="cuda", dtype=dtype), torch.tensor(reff, device="cuda"), q,
                      S=torch.tensor(S, device="cuda"), convention="larch").double().cpu().numpy()
    ang = np.unwrap(np.angle(cc), axis=1)
    ref = (np.sqrt(np.abs(cc) ** 2 + 1e-30) @ S.T) * np.sin(ang @ S.T + 2 * q[None] * reff[:, None])
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()
