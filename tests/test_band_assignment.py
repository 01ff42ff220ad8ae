"""The wavefronts of the energy bands (tables._assign): a valid assignment whose largest total is the one returned, never
worse than longest-processing-time first, the optimum for few bands; nothing when the bound cannot be met."""
import itertools

import numpy as np
import pytest

from feffgpu_amd import tables as T


def _lpt(costs):
    load = [0.0] * T.WAVES
    for c in sorted(costs, reverse=True):
        load[int(np.argmin(load))] += c
    return max(load)


@pytest.mark.parametrize("nb", [1, 2, 4, 5, 6, 7, 16])
@pytest.mark.parametrize("seed", range(5))
def test_assignment(nb, seed):
    costs = [float(c) for c in np.random.default_rng(seed).integers(8, 45, nb)]
    wave, span = T._assign(costs)
    tot = [sum(c for c, w in zip(costs, wave) if w == k) for k in range(T.WAVES)]
    assert len(wave) == nb and span == max(tot) and span <= _lpt(costs)
    if nb <= 6:
        assert span == min(max(sum(c for c, w in zip(costs, a) if w == k) for k in range(T.WAVES))
                           for a in itertools.product(range(T.WAVES), repeat=nb))
    assert T._assign(costs, below=span) == (None, np.inf)
