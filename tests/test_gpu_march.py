"""Statistics and properties where the marching kernels walk 1, 2, 4, 8 and 16 cells
(csrc/lpt_kernels.hip: march_of), with lines that are no multiple of the walk: the
check, tolerances and oracle of test_gpu_output_edges.py."""
import pytest

from test_gpu_output_edges import test_statistics_and_properties as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,n", [(40, 300), (59, 100), (67, 500), (85, 64), (103, 200), (126, 129)])
def test_walks(nc, n):
    check(nc, n)
