"""The persistent head kernel over fp8 weights at 17 to 32 rows, which it takes from 131072 features on: tests/test_head_fp8_gpu.py's comparison."""
import pytest

from test_head_fp8_gpu import test_head as compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(17, 131072), (32, 131104), (32, 131040)])
def test_few_rows(M, N):
    compare(M, N, 1024)
