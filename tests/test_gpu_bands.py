"""The defect kernel at the edges of its split into row bands: grids of at most
128 columns, which put several bands into a workgroup (with and without idle
threads), the first that do not, single rows; checks and tolerances of the same
kernel's comparison with the oracle."""
import pytest

import test_gpu_stream as S
from test_gpu_stream import lib  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 7), (4, 130), (85, 84), (128, 10), (130, 34), (256, 5), (300, 33)])
def test_defect_bands(lib, prec, nx, ny):  # noqa: F811
    S.test_defect_matches_oracle(lib, prec, nx, ny, 1 / nx, 1.3 / ny, 1.9, -2.4)
