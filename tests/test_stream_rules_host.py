"""Which products over fp32 rows and bf16 weights the streaming kernel takes (mi_gemm_any_streams): where it was measured slower than the tile kernels it
stays out."""
import pytest

from nanovllm import _C

takes = lambda rows, N, K, groups=0: bool(_C.lib.mi_gemm_any_streams(rows, N, K, groups))


@pytest.mark.parametrize("rows,N,K", [(24, 18432, 64), (17, 32768, 256), (24, 12288, 2048), (32, 9216, 4096), (17, 16384, 8192), (9, 12288, 4096), (33, 6160, 2048),
                                      (49, 4112, 64), (65, 64, 64), (8, 64, 64), (9, 64, 96)])
def test_slower_shapes_stay_out(rows, N, K):
    assert not takes(rows, N, K)


@pytest.mark.parametrize("rows,N,K", [(24, 18432, 512), (16, 32768, 64), (24, 12288, 1024), (32, 8192, 4096), (17, 16384, 4096), (9, 12288, 2048), (48, 6144, 2048),
                                      (64, 4096, 64), (48, 4224, 2048), (9, 1, 64)])
def test_faster_shapes_are_taken(rows, N, K):
    assert takes(rows, N, K)


def test_groups():
    assert takes(640, 768, 2048, 64) and not takes(641, 768, 2048, 64)
    assert takes(512, 2048, 768, 64) and not takes(513, 2048, 768, 64)
    assert not takes(944, 768, 256, 128) and takes(944, 256, 768, 128) and takes(96, 512, 256, 32)
