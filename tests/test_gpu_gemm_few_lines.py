"""The GEMM for a few rows at the shallower depths it also takes (`gemm_few_kernel`): around 1024 and 3072, where fewer K-tiles
than the eight waves hold in flight leave requests past the end, rows and columns at the edges of its blocks."""
import pytest

from test_gpu_gemm_few import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mn", [(1, 1), (16, 17), (9, 4096), (16, 4097)])
@pytest.mark.parametrize("K", [1008, 1024, 1040, 1920, 2032])
def test_sixteen_rows(mn, K):
    _check(*mn, K)


@pytest.mark.parametrize("mn", [(17, 1), (31, 2047), (32, 33), (32, 4096)])
@pytest.mark.parametrize("K", [3056, 3072, 3088, 4096, 5120])
def test_thirty_two_rows(mn, K):
    _check(*mn, K)
