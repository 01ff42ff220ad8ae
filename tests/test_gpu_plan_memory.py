"""What a plan holds for its adjoint: at most HELD_BYTES; a call that runs in more takes it for its own time. The gradient
is the same with a workspace of the call's own, held, or too small for the lanes: the FP64 sums over the energies may be
split differently, 1e-12 of the largest component."""
import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
Q = np.arange(0.0, 18.0001, 0.05)


def _plan(repeat=1, prec=32):
    from feffgpu_amd.paths import PathPlan
    pos0, box = W.lattice("bcc", 2.87, 4)
    pos = W.displaced(pos0, 0.07, 3)
    pl = W.concat([W.enumerate_paths(pos, a, np.full(len(pos), 2), 4.6, 4, box=box, segment=i, nmax=4)
                   for i, a in enumerate((0, 17))], 4)
    t = lambda a: np.concatenate([a] * repeat)
    plan = PathPlan(str(GOLDEN / "validation" / "A018" / "phase.pad"), Q, t(pl.atoms), t(pl.nleg), t(pl.absorber),
                    t(pl.ipots), t(pl.deg), segment=t(pl.segment), nseg=2, cell=float(box[0]), precision=prec)
    return plan, torch.tensor(pos, device="cuda"), torch.tensor(np.random.default_rng(1).normal(size=(2, len(Q))),
                                                               device="cuda")


def _close(a, b):
    return float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


def test_a_long_list_holds_no_more():
    from feffgpu_amd.paths import HELD_BYTES
    plan, p, g = _plan()
    plan.forward(p, keep=True)
    want = plan.backward(p, g, kept=True)
    assert plan._call_bytes == 0 and plan.workspace.numel() <= HELD_BYTES
    r = 120_000 // plan.npath
    plan, p, g = _plan(r)
    assert plan.workspace.numel() <= HELD_BYTES < plan._call_bytes
    plan.forward(p, keep=True)
    plan.backward(p, g)
    before = torch.cuda.memory_allocated()
    got = plan.backward(p, g, kept=True)
    assert torch.cuda.memory_allocated() - before <= got.numel() * 8 + 512
    assert _close(got / r, want)


@pytest.mark.parametrize("prec", [32, 64])
def test_the_calls_workspace(monkeypatch, prec):
    from feffgpu_amd import paths
    from feffgpu_amd.graph import CapturedStep
    plan, p, g = _plan(40, prec)
    assert plan._call_bytes == 0
    plan.forward(p, keep=True)
    want = [plan.backward(p, g, kept=True), plan.backward(p, g)]
    monkeypatch.setattr(paths, "HELD_BYTES", 1 << 20)
    plan, p, g = _plan(40, prec)
    held = plan.workspace.numel()
    assert plan._call_bytes > held
    plan.forward(p, keep=True)
    assert all(_close(a, b) for a, b in zip([plan.backward(p, g, kept=True), plan.backward(p, g)], want))
    step = CapturedStep(plan, len(p))
    for k in range(3):
        seg, grad = step(p, g)
        assert _close(grad, want[0])
        moved = p + 0.01 * (k + 1)
        plan.forward(moved, keep=True)
        plan.backward(moved, g, kept=True)
        torch.cuda.synchronize()
    plan._call_bytes = 1 << 50          # no device has that: the held workspace, in chunks
    plan.forward(p, keep=True)
    assert all(_close(a, b) for a, b in zip([plan.backward(p, g, kept=True), plan.backward(p, g)], want))
