"""Lists so long that a kernel with many threads per path would pass 2^32 threads of a launch: every path is evaluated.
The lists repeat one path, so every row equals that of a short list."""
import ctypes

import numpy as np
import pytest
import torch

from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
PHASE = GOLDEN / "validation" / "A018" / "phase.pad"


def _room(nbytes):
    if torch.cuda.mem_get_info()[0] < nbytes:
        pytest.skip("needs %d GB of device memory" % (nbytes >> 30))


def test_importance_of_more_than_2_29_paths():
    """Eight lanes per path."""
    from feffgpu_amd.pathfinder import GPUPathFinder
    P = (1 << 29) + 3
    _room(48 << 30)
    fd = GPUPathFinder(str(PHASE))
    one = torch.tensor([[[0.0, 0.0, 0.0], [0.3, 2.1, 0.9]]], device="cuda")
    ip = torch.tensor([[0, 1]], device="cuda")
    want, rt = fd._importance(one, ip)
    got, rtot = fd._importance(one.expand(P, -1, -1).contiguous(), ip.expand(P, -1).contiguous())
    other = int(torch.count_nonzero(got != want)) + int(torch.count_nonzero(rtot != rt))
    assert other == 0


@pytest.mark.parametrize("P", [(1 << 26) + 5, (1 << 27) + 9])
def test_single_scattering_list_of_more_than_2_26_paths(P):
    """One wavefront per path in the fine grid's own kernel; 32 threads per path in the energies'."""
    from feffgpu_amd import _native as N
    from feffgpu_amd.paths import PathPlan
    q = np.linspace(0.0, 0.6, 40)
    _room(64 << 30)
    one = PathPlan(str(PHASE), q, [[1]], [2], [0], [[0, 1]], [1.0], precision=32, device="cuda")
    pos = torch.tensor([[0.0, 0.0, 0.0], [0.4, 1.9, 1.1]], device="cuda", dtype=torch.float64)
    want = one.forward(pos)[1]
    assert one.nk >= 2 * one.tables[0].E + 3            # a row holds what a long list leaves there
    t = {k: getattr(one, k).expand((P,) + getattr(one, k).shape[1:]).contiguous()
         for k in ("atoms_t", "nleg_t", "absorber_t", "ipots_t", "deg_t", "edge_t")}
    ps = one._paths_struct(pos)
    ps.npath = P
    ps.atoms, ps.nleg, ps.absorber, ps.ipots, ps.deg, ps.edge = (v.data_ptr() for v in t.values())
    chi = torch.empty(P, one.nk, device="cuda", dtype=torch.float32)
    reff = torch.empty(P, device="cuda", dtype=torch.float64)
    i = lambda *v: (ctypes.c_int32 * len(v))(*v)
    N.check(N.lib().fm_chi_paths(one.edge_array, 1, ps, one.grid, 32, 2, None, 1, i(0, P), i(int(one.buckets.kind[0])),
                                 i(0), i(2), 0, None, None, None, chi.data_ptr(), reff.data_ptr(), None,
                                 N.stream_of(one.device)), "fm_chi_paths")
    other = int(torch.count_nonzero(chi != want)) + int(torch.count_nonzero(reff != one.reff))
    assert float(want.abs().max()) > 0 and other == 0
