"""The buckets of a path list on side streams: the results are those of the buckets one after the other, bit for bit
(the same launches on the same data), in eager calls, with a workspace too small for the lanes, with buckets of 7 and 8
legs, under capture with replays between eager calls, and from two plans in two threads; also the lanes' sets are given
back and taken again."""
import gc
import threading

import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
Q = np.arange(0.0, 18.0001, 0.05)


def _plan(seed, legs=5, prec=32, rmax=4.4):
    from feffgpu_amd.paths import PathPlan
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = W.displaced(pos0, 0.07, seed)
    ipot = np.full(len(pos), 1)
    pl = W.concat([W.enumerate_paths(pos, a, ipot, rmax, legs, box=box, segment=i, nmax=legs)
                   for i, a in enumerate((5, 77, 20))], legs)
    rng = np.random.default_rng(seed)
    plan = PathPlan([str(GOLDEN / "validation" / c / "phase.pad") for c in ("A014", "A018")], Q, pl.atoms, pl.nleg,
                    pl.absorber, pl.ipots, pl.deg, segment=pl.segment, nseg=3, edge=(pl.absorber == 77).astype(int),
                    cell=float(box[0]), precision=prec, device="cuda")
    g = torch.tensor(rng.normal(size=(3, len(Q))), device="cuda")
    return plan, torch.tensor(pos, device="cuda"), g


def _run(plan, p, g):
    seg = plan.forward(p, keep=True)[0].clone()
    return seg, plan.backward(p, g, kept=True).clone(), plan.backward(p, g).clone()


def _l001(prec):
    """FEFF's list of 2-8 legs around one absorber."""
    from feffgpu_amd.feffio import read_paths_dat
    from feffgpu_amd.paths import PathPlan
    d = GOLDEN / "validation" / "L001"
    paths = read_paths_dat(d / "paths.dat")
    nmax = max(p.nleg for p in paths)
    pos, atoms = [np.zeros(3)], []
    for x in paths:
        atoms.append(list(range(len(pos), len(pos) + x.nleg - 1)) + [0] * (nmax - x.nleg))
        pos += list(x.coords[1:])
    plan = PathPlan(str(d / "phase.pad"), Q, np.array(atoms), np.array([x.nleg for x in paths]),
                    np.zeros(len(paths), int), np.array([list(x.ipots) + [0] * (nmax - x.nleg) for x in paths]), np.array([x.deg for x in paths]),
                    nseg=1, precision=prec, device="cuda")
    return plan, torch.tensor(np.array(pos), device="cuda"), torch.ones(1, len(Q), device="cuda", dtype=torch.float64)


@pytest.mark.parametrize("legs,prec", [(3, 32), (4, 64), (5, 32), (8, 32), (8, 64)])
def test_same_as_one_after_the_other(legs, prec):
    plan, p, g = _l001(prec) if legs == 8 else _plan(31, legs, prec)
    assert len(plan.buckets.kind) >= 4 and plan._overlap
    with_lanes = [_run(plan, p, g) for _ in range(3)]
    full = plan.workspace
    from feffgpu_amd import _native as N
    plan.workspace = full[:int(N.lib().fm_backward_workspace_bytes(prec, plan.nmax, 16)) + (64 << 10)]
    small = _run(plan, p, g)
    plan.workspace = full
    lanes, plan._overlap = plan._overlap, None
    alone = _run(plan, p, g)
    plan._overlap = lanes
    for r in with_lanes:
        assert all(torch.equal(a, b) for a, b in zip(r, alone))
    assert torch.equal(small[0], alone[0])
    for a, b in zip(small[1:], alone[1:]):     # chunks: the FP64 sums over the energies may be split differently
        assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


def test_captured_step_and_eager_calls_between_replays():
    plan, p, g = _plan(7)
    want = _run(plan, p, g)
    static = p.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _run(plan, static, g)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _run(plan, static, g)
    moved = p + 0.01
    want2 = _run(plan, moved, g)
    for x, w in ((p, want), (moved, want2), (p, want)):
        static.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, w))
        assert all(torch.equal(a, b) for a, b in zip(_run(plan, moved, g), want2))


def test_two_threads_and_returned_sets():
    want, got = {}, {}
    for s in (1, 2):
        plan, p, g = _plan(s)
        want[s] = _run(plan, p, g)
        torch.cuda.synchronize()
        del plan
        gc.collect()

    def work(s):
        with torch.cuda.stream(torch.cuda.Stream()):
            plan, p, g = _plan(s)
            for _ in range(5):
                got[s] = _run(plan, p, g)
            torch.cuda.current_stream().synchronize()
    th = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    [t.start() for t in th]
    [t.join() for t in th]
    for s in (1, 2):
        assert all(torch.equal(a, b) for a, b in zip(got[s], want[s]))


def test_no_room_for_the_lanes(monkeypatch):
    """A device without room for a region per lane gets the smaller workspace and the same results."""
    from feffgpu_amd import _native as N
    plan, p, g = _plan(5)
    want, real = _run(plan, p, g), N.backward_workspace

    def full(*a, at_least=0, **k):
        if at_least:
            raise torch.cuda.OutOfMemoryError("no room")
        return real(*a, **k)
    monkeypatch.setattr(N, "backward_workspace", full)
    plan, p, g = _plan(5)
    assert all(torch.equal(a, b) for a, b in zip(_run(plan, p, g), want))
