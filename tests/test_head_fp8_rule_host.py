"""Which fp8 heads go to the persistent kernel, as the number of candidates that each row's pick is made from shows it (mi_gemm_pick_groups)."""
import pytest

from nanovllm import _C

groups = lambda M, N, K: _C.lib.mi_gemm_pick_groups(M, N, K, 1)


@pytest.mark.parametrize("M,N,K,want", [(24, 65536, 1024, 65536 // 32), (32, 114688, 1024, 114688 // 32), (17, 131072, 1024, 1024), (32, 151936, 1024, 1024), (16, 151936, 1024, 151936 // 32),
                                        (33, 65536, 1024, 512), (200, 65536, 1024, 512), (33, 65536, 896, 512), (32, 151936, 896, 151936 // 32)])
def test_persistent_workgroups(M, N, K, want):
    assert groups(M, N, K) == want
