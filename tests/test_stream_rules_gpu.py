"""The streaming kernel with two feature tiles per workgroup from 4097 features on (csrc/gemm_any.hip), against float64 over the rounded operands: the
first sizes of that form, features that end inside a workgroup's first and second tile (bound: tests/test_gemm_any_stream_gpu.py)."""
import pytest
import torch

from nanovllm import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [9, 17, 33, 48])
@pytest.mark.parametrize("N,K", [(4096, 192), (4097, 192), (4110, 64), (4128, 640), (5119, 128)])
def test_two_tiles(M, N, K):
    from nanovllm import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda", generator=g)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    assert _C.lib.mi_gemm_any_streams(M, N, K, 0)
    out = torch.full((M + 1, N + 4), 7.0, device="cuda")
    ops.gemm_any(x, w, out=out[:M, :N])
    xr = x.bfloat16().double()
    assert bool(((out[:M, :N].double() - xr @ w.double().T).abs() <= (K + 16) * 2.0 ** -24 * (xr.abs() @ w.double().abs().T) + 1e-6).all())
    assert bool((out[M] == 7.0).all() and (out[:, N:] == 7.0).all())
