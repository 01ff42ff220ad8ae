"""MultipleScattering evaluates the list of its last enumeration: further enumerations on one object (moved
atoms; another number of copies and absorbers; the first frames again) give the rows, the subset's chi and the gradient of a
fresh object, bit for bit."""
import numpy as np
import pytest
import torch

from feffgpu_amd import workloads as W
from fixtures import GOLDEN

pytestmark = pytest.mark.gpu
K = np.round(np.arange(0.0, 16.0 + 1e-9, 0.05), 10)


def _object():
    from feffgpu_amd.forward import MultipleScattering
    return MultipleScattering(str(GOLDEN / "validation" / "A018" / "phase.pad"), K, 3.0, W.lattice("bcc", 2.87, 4)[1][0],
                              rmax=4.6, critpw=2.0, nlegmax=4)


def _frames(C, sigma, seed):
    pos0, _ = W.lattice("bcc", 2.87, 4)
    return np.stack([W.displaced(pos0, sigma, (seed, c)) for c in range(C)])


def _evaluate(ms, frames, absorbers):
    flat = torch.tensor(frames.reshape(-1, 3), device="cuda")
    ms.enumerate(frames, absorbers=absorbers)
    rows = ms.full_pass(flat).clone()
    some = ms.chi_absorbers(flat, ms.abs_atoms[:2]).detach()
    return rows, some, ms.full_gradient(flat, lambda m: (m ** 2).sum())


def test_every_enumeration_has_its_own_plan():
    held = _object()
    jobs = [(_frames(2, 0.05, 1), [0, 9]), (_frames(2, 0.20, 2), [0, 9]), (_frames(3, 0.1, 3), [5, 17, 40]),
            (_frames(2, 0.05, 1), [0, 9])]
    for frames, ab in jobs:
        got, want = _evaluate(held, frames, ab), _evaluate(_object(), frames, ab)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert float(want[0].abs().max()) > 0
