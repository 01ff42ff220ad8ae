"""The adjoint's streams with 8 (path, scatterer) units per workgroup (4096 to 8191 units in a launch) and a partial last
workgroup: rows of the call equal calls on one path (FP64 sums over at most 60 energies split differently: 1e-11 of the
path's largest component), and FP32 equals FP64 to 1e-4, as for the other numbers of units."""
import pytest

from test_gpu_adjoint_sizes import test_rows_equal_single_paths as _rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case,nleg,npath", [("validation/A018", 3, 2051), ("validation/L001", 4, 1501),
                                             ("validation/L001", 5, 1101), ("validation/L001", 6, 901),
                                             ("validation/A014", 3, 3001), ("validation/A014", 4, 1501)])
def test_eight_units(case, nleg, npath):
    assert 4096 <= npath * (nleg - 1) < 8192 and npath % 8
    _rows(case, nleg, npath)
