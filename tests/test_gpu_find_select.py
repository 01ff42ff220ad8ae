"""The finder's filter as row numbers (fm_find_select), the kept rows moved up (fm_find_compact) and the reference
importances (fm_find_ref) against the same selections in torch and numpy: bytes are equal. Sizes at the edges of the
scan's blocks (4096) and of a thread block; nothing kept, everything kept, some kept; the finder with its passes cut
into pieces."""
import ctypes

import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu


def _rows(P, nleg, rng, A):
    return dict(atoms=torch.tensor(rng.integers(0, 99, (P, nleg - 1)), device="cuda"),
                coords=torch.tensor(rng.normal(size=(P, nleg, 3)), device="cuda", dtype=torch.float32),
                ipots=torch.tensor(rng.integers(0, 3, (P, nleg)), device="cuda"),
                deg=torch.tensor(rng.integers(1, 3, P), device="cuda", dtype=torch.float32),
                slot=torch.tensor(np.sort(rng.integers(0, A, P)), device="cuda", dtype=torch.int32))


@pytest.mark.parametrize("P", [0, 1, 255, 4095, 4096, 4097, 20000])
@pytest.mark.parametrize("nleg", [2, 3, 9])
@pytest.mark.parametrize("critpw", [0.0, 55.0, 1e9])
def test_select_and_compact(P, nleg, critpw):
    from feffgpu_amd import _native as N
    from feffgpu_amd.pathfinder import GPUPathFinder, _ROWS
    L, A = N.lib(), 7
    rng = np.random.default_rng(P + nleg)
    o = _rows(P, nleg, rng, A)
    xp = torch.tensor(rng.random(P), device="cuda", dtype=torch.float32)
    ref = torch.tensor(1 + rng.random(A), device="cuda", dtype=torch.float32)
    st = N.stream_of(o["deg"].device)
    pos = torch.empty(P, dtype=torch.int64, device="cuda")
    tot = torch.empty(1, dtype=torch.int64, device="cuda")
    ws = torch.empty(int(L.fm_scan_workspace_bytes(P)), dtype=torch.uint8, device="cuda")
    N.check(L.fm_find_select(P, o["deg"].data_ptr(), xp.data_ptr(), o["slot"].data_ptr(), ref.data_ptr(), critpw,
                             pos.data_ptr(), tot.data_ptr(), ws.data_ptr(), ws.numel(), st), "select")
    sel = ((100 * o["deg"]) * xp) / ref[o["slot"].long()] >= np.float32(critpw)
    n = int(sel.sum())
    assert int(tot) == n and torch.equal(pos, torch.cumsum(sel, 0) - sel.long())
    t = {k: torch.empty((n,) + v.shape[1:], dtype=v.dtype, device="cuda") for k, v in o.items()}
    x = torch.empty(n, dtype=torch.float32, device="cuda")
    if n == 0:          # no rows, no buffers to move them to
        return
    N.check(L.fm_find_compact(P, nleg, pos.data_ptr(), tot.data_ptr(), ctypes.byref(GPUPathFinder._out_struct(o)),
                              xp.data_ptr(), ctypes.byref(GPUPathFinder._out_struct(t)), x.data_ptr(), st), "compact")
    assert torch.equal(x, xp[sel]) and all(torch.equal(t[k], o[k][sel]) for k in _ROWS)


@pytest.mark.parametrize("merged", [0, 1])
def test_reference_importance(merged):
    from feffgpu_amd import _native as N
    rng = np.random.default_rng(3)
    A = 9
    slot = np.sort(rng.choice([0, 1, 3, 4, 8], 300))          # absorbers without paths, too
    d = rng.integers(20, 60, 300).astype(np.float32)           # many equal lengths: the first one counts
    xp, deg = rng.random(300).astype(np.float32), rng.integers(1, 5, 300).astype(np.float32)
    nc = np.array([1, 5, 0, 2, 1, 0, 0, 0, 3], np.int32)
    ref = torch.empty(A, dtype=torch.float32, device="cuda")
    t = [torch.tensor(v, device="cuda") for v in (slot.astype(np.int32), d, xp, deg, nc)]
    N.check(N.lib().fm_find_ref(A, 300, *(v.data_ptr() for v in t), merged, ref.data_ptr(), N.stream_of(ref.device)),
            "fm_find_ref")
    want = np.ones(A, np.float32)
    for b in range(A):
        m = np.nonzero(slot == b)[0]
        if len(m):
            k = m[np.argmin(d[m])]
            want[b] = xp[k] * deg[k] if merged and nc[b] > 1 else xp[k]
    assert np.array_equal(ref.cpu().numpy(), want)


@pytest.mark.parametrize("critpw", [0.0, 3.0])
def test_pieces_of_the_filter(critpw, monkeypatch):
    from feffgpu_amd import pathfinder as F
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = W.displaced(pos0, 0.07, 31)
    fd = F.GPUPathFinder(str(GOLDEN / "validation" / "A018" / "phase.pad"), rmax=5.0, nlegmax=4, critpw=critpw,
                         merge_degenerate=False)
    ip = np.full(len(pos), 2)
    whole, ref = fd.enumerate_many(pos, float(box[0]), [0, 9, 77], ip)
    monkeypatch.setattr(F, "SELECT_MAX", 100)
    cut, ref2 = fd.enumerate_many(pos, float(box[0]), [0, 9, 77], ip)
    assert np.array_equal(ref, ref2) and whole.keys() == cut.keys()
    for n in whole:
        assert all(torch.equal(whole[n][k], cut[n][k]) for k in whole[n])
    for bad in ([-1, 3], [len(pos)], torch.tensor([0, 10 ** 6], device="cuda")):
        with pytest.raises(ValueError, match="absorber index"):
            fd.enumerate_many(pos, float(box[0]), bad, ip)


@pytest.mark.parametrize("npath", [1, 7, 32, 33])
@pytest.mark.parametrize("nleg", range(2, 10))
def test_importance_of_every_number_of_legs(nleg, npath):
    """8 lanes per path, 32 paths per block. FP64 formula on the float32 tables and bins: a chain of up to 9 products and
    divisions and an exponential per energy, 75 terms of one sign: 1e-5."""
    from feffgpu_amd.pathfinder import GPUPathFinder, NBETA
    fd = GPUPathFinder(str(GOLDEN / "validation" / "A018" / "phase.pad"))
    rng = np.random.default_rng(10 * nleg + npath)
    c = (rng.uniform(-3, 3, (npath, nleg, 3)) + 2.0 * np.arange(nleg)[None, :, None]).astype(np.float32)
    c[:, 0] = 0
    ip = rng.integers(0, fd.fbeta.shape[1], (npath, nleg))
    got, rtot = (v.cpu().numpy() for v in fd._importance(c, ip))
    leg = np.roll(c, -1, 1) - c
    ri = np.sqrt((leg * leg).sum(-1))
    u = leg / ri[..., None]
    cosv = (u[:, :-1] * u[:, 1:]).sum(-1).astype(np.float32)
    a = np.abs(cosv)
    n = np.floor(a / np.float32(0.025))
    n = (n + (a - n * np.float32(0.025) > np.float32(0.0125))) * np.where(cosv < 0, -1, 1)
    k = np.clip(n.astype(int) + NBETA, 0, 2 * NBETA)
    cmax = np.maximum(np.abs((u[:, -1] * u[:, 0]).sum(-1)), 0.3).astype(float)
    fb, ck, xl, w = (v.double().cpu().numpy() for v in (fd.fbeta, fd.cksp, fd.xlam, fd.trap))
    ri = ri.astype(float)
    want = np.zeros(npath)
    for i, e in enumerate(range(fd.ik0, len(ck))):
        crit = cmax / (ri[:, -1] * ck[e])
        for j in range(nleg - 1):
            crit = crit * fb[e, ip[:, j + 1], k[:, j]] / (ri[:, j] * ck[e])
        want += np.abs(crit * np.exp(-ri.sum(1) / xl[e])) * w[i]
    assert np.allclose(got, want, rtol=1e-5, atol=0) and np.allclose(rtot, ri.sum(1), rtol=1e-6)
