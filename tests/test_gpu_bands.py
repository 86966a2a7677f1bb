"""The row-mapped kernels of a block step (defect, lifting right-hand side and
update) at the edges of their split into row bands: grids of at most 128
columns, which put several bands into a workgroup (one column to 128, with and
without idle threads), the first that do not, and single rows and columns;
checks and tolerances of the same kernels' comparison with the oracle."""
import numpy as np
import pytest

import test_gpu_stream as S
from test_gpu_stream import lib  # noqa: F401

pytestmark = pytest.mark.gpu

SIZES = [(2, 2), (3, 7), (4, 130), (85, 84), (128, 10), (130, 34), (256, 5), (300, 33)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_bands(lib, prec, nx, ny):  # noqa: F811
    grid = (nx, ny, 1 / nx, 1.3 / ny, 1.9, -2.4)
    S.test_defect_matches_oracle(lib, prec, *grid)
    S.test_lift_rhs_matches_oracle(lib, prec, True, True, *grid)
    S.test_lift_rhs_matches_oracle(lib, prec, False, False, *grid)
    S.test_lift_apply_matches_oracle(lib, prec, False, *grid)
