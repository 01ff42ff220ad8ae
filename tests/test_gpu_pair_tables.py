"""The adjoint of single scattering from pair tables.

* fm_pair_chi_grad: gbin = tables @ gchi / div for tables of both types, several potentials in any order of their rows;
  a sum of at most 361 FP64 products, 1e-13 of the sum of their absolute values; other rows stay untouched.
* fm_pair_histogram_grad in every kind of cell against autograd through torch's FP64 distances of all pairs: each
  component a sum of n terms of one (gb1 - gb0) / dr each, 1e-10 of the largest component.
* More pairs than the fixed-point bins take (the histograms of chunks of configurations summed in FP64): chi and gradient
  of one call, 1e-12 of the largest value.
* The tables may be changed in place between a forward call and its gradient, which is that of the tables as they were."""
import ctypes

import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
Q = np.arange(0, 18.0001, 0.05)


@pytest.fixture()
def tables():
    from feffgpu_amd.pairs import PairTables
    pos0, box = W.lattice("bcc", 2.87, 5)
    pt = PairTables(str(GOLDEN / "validation" / "A018" / "phase.pad"), Q, box=float(box[0]), rmax=5.6, dr=0.01, ms=False)
    pt.ipot = torch.tensor(np.random.default_rng(3).integers(1, pt.npot, len(pos0)), device="cuda")
    return pt, pos0


@pytest.mark.parametrize("nr,nk", [(2, 1), (5, 63), (411, 64), (410, 361)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_bin_gradient(dtype, nr, nk):
    from feffgpu_amd import _native as N
    rng = np.random.default_rng(nr + nk)
    rows = [3, 1]
    T = [torch.tensor(rng.normal(size=(nr, nk)), device="cuda", dtype=dtype) for _ in rows]
    g = torch.tensor(rng.normal(size=nk), device="cuda")
    gbin = torch.full((5, nr), 7.0, device="cuda", dtype=torch.float64)
    N.check(N.lib().fm_pair_chi_grad(2, (ctypes.c_void_p * 2)(*[t.data_ptr() for t in T]), (ctypes.c_int32 * 2)(*rows),
                                     32 if dtype == torch.float32 else 64, nr, nk, g.data_ptr(), 37.0, gbin.data_ptr(),
                                     N.stream_of(g.device)), "fm_pair_chi_grad")
    for t, r in zip(T, rows):
        want, scale = t.double() @ g / 37.0, t.double().abs() @ g.abs() / 37.0
        assert bool(((gbin[r] - want).abs() <= 1e-13 * scale).all())
    assert bool((gbin[[0, 2, 4]] == 7.0).all())


@pytest.mark.parametrize("n", [3, 17, 200])
@pytest.mark.parametrize("kind", ["cubic", "general", "oblique", "cluster"])
def test_position_gradient_in_every_cell(tables, kind, n):
    from feffgpu_amd import _native as N
    pt, _ = tables
    rng = np.random.default_rng(n)
    L = 2.2 * pt.rmax
    cell = {"cubic": L, "general": np.diag([L, 0.9 * L, 1.3 * L]), "cluster": None,
            "oblique": np.array([[L, 0, 0], [0.3 * L, 0.95 * L, 0], [-0.2 * L, 0.25 * L, 0.9 * L]])}[kind]
    g, npot = pt._grid(cell), 3
    pos = torch.tensor(rng.uniform(0, 0.3 * L if n == 3 else 0.6 * L, (n, 3)), device="cuda")
    ip = torch.tensor(rng.integers(-1, npot + 1, n), device="cuda", dtype=torch.int32)
    gbin = torch.tensor(rng.normal(size=(npot, pt.nr)), device="cuda")
    got = torch.empty(1, n, 3, device="cuda", dtype=torch.float64)
    N.check(N.lib().fm_pair_histogram_grad(1, n, pos.data_ptr(), ip.data_ptr(), npot, ctypes.byref(g), gbin.data_ptr(),
                                           got.data_ptr(), N.stream_of(pos.device)), "fm_pair_histogram_grad")
    x = pos.clone().requires_grad_(True)
    rel = x[None] - x[:, None]
    if cell is not None:
        c = torch.tensor(np.eye(3) * cell if np.ndim(cell) == 0 else cell, device="cuda")
        f = rel.detach() @ torch.linalg.inv(c)
        rel = rel - torch.round(f) @ c
    r2 = (rel ** 2).sum(-1)
    a, j = torch.nonzero((r2 <= pt.rmax ** 2) & (r2 > 1e-6) & (ip[None] >= 0) & (ip[None] < npot), as_tuple=True)
    u = (torch.sqrt(r2[a, j]) - pt.r0) / pt.dr
    i0 = torch.floor(u.detach()).clamp(0, pt.nr - 2).long()
    f = (u - i0).clamp(0, 1)
    p = ip[j].long()
    (want,) = torch.autograd.grad(((1 - f) * gbin[p, i0] + f * gbin[p, i0 + 1]).sum(), x)
    assert len(a) > 0 and float((got[0] - want).abs().max()) <= 1e-10 * float(want.abs().max())


def test_chunks_of_configurations(tables, monkeypatch):
    from feffgpu_amd import pairs
    pt, pos0 = tables
    n = len(pos0)
    pos = torch.tensor(np.stack([W.displaced(pos0, 0.1, (8, c)) for c in range(5)]), device="cuda", requires_grad=True)
    w = torch.linspace(-1, 1, len(Q), device="cuda", dtype=torch.float64)
    out = []
    for pairs_per_call in (pairs._BIN_PAIRS, 2 * n * (n - 1) + 1, 2):
        monkeypatch.setattr(pairs, "_BIN_PAIRS", pairs_per_call)
        chi = pt.single_scattering(pos)
        out.append((chi.detach(), torch.autograd.grad((chi * w).sum(), pos)[0]))
    for chi, g in out[1:]:
        assert float((chi - out[0][0]).abs().max()) <= 1e-12 * float(out[0][0].abs().max())
        assert torch.equal(g, out[0][1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_tables_changed_after_the_forward(tables, dtype):
    pt, pos0 = tables
    pt.tables = {p: t.to(dtype) for p, t in pt.tables.items()}
    pos = torch.tensor(W.displaced(pos0, 0.1, 8)[None], device="cuda", requires_grad=True)
    (want,) = torch.autograd.grad(pt.single_scattering(pos).sum(), pos)
    chi = pt.single_scattering(pos)
    for t in pt.tables.values():
        t.mul_(0.5)
    (got,) = torch.autograd.grad(chi.sum(), pos)
    assert torch.equal(got, want)
    (half,) = torch.autograd.grad(pt.single_scattering(pos).sum(), pos)
    assert float((half - 0.5 * want).abs().max()) <= 1e-12 * float(want.abs().max())
