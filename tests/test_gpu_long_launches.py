"""Lists so long that a kernel with many threads per path would pass 2^32 threads of a launch: every path is evaluated.
The lists repeat one path, so every row equals that of a short list."""
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
