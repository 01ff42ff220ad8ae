"""fm_find_filter's flags are the rows that fm_find_select keeps."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 256, 4097])
@pytest.mark.parametrize("critpw", [0.0, 55.0, 1e9])
def test_flags_are_the_selection(P, critpw):
    from feffgpu_amd import _native as N
    L = N.lib()
    rng = np.random.default_rng(P)
    deg, xp, ref = (torch.tensor(v, device="cuda", dtype=torch.float32)
                    for v in (rng.integers(1, 3, P), rng.random(P), 1 + rng.random(5)))
    slot = torch.tensor(np.sort(rng.integers(0, 5, P)), device="cuda", dtype=torch.int32)
    st = N.stream_of(deg.device)
    keep = torch.empty(P, dtype=torch.uint8, device="cuda")
    N.check(L.fm_find_filter(P, deg.data_ptr(), xp.data_ptr(), slot.data_ptr(), ref.data_ptr(), critpw, keep.data_ptr(),
                             st), "fm_find_filter")
    pos = torch.empty(P + 1, dtype=torch.int64, device="cuda")
    ws = torch.empty(int(L.fm_scan_workspace_bytes(P)), dtype=torch.uint8, device="cuda")
    N.check(L.fm_find_select(P, deg.data_ptr(), xp.data_ptr(), slot.data_ptr(), ref.data_ptr(), critpw, pos.data_ptr(),
                             pos[P:].data_ptr(), ws.data_ptr(), ws.numel(), st), "fm_find_select")
    assert torch.equal(keep.long(), pos[1:] - pos[:-1])
