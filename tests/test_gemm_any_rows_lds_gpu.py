"""Two to eight rows of true fp32 by many features of bf16 weights (the rows in LDS): against 64 bits; features that are no whole fours and no
whole workgroups, rows of a wider buffer, activations, and what the rule leaves where it was (a K of 520, rows off 16 bytes, one row)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [512, 1024, 2048, 4096, 520])
@pytest.mark.parametrize("N", [4094, 4096, 6145, 8192, 16421, 33000])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 7, 8])
def test_rows(M, N, K):
    from nanovllm import _C, ops

    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    wide = torch.randn(M, K + 8, device="cuda", generator=g)
    w = (torch.randn(N, K, device="cuda", generator=g) / 16).bfloat16()
    bias = torch.randn(N, device="cuda", generator=g)
    for x in (wide[:, 4:K + 4], wide[:, 1:K + 1]):
        z, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        room = (K // 64 + 8) * 2.0 ** -24 * mag + 2.0 ** -23 * z.abs()   # a lane's fused steps, the lanes' tree, the result
        out = torch.full((M + 1, N + 4), 7.0, device="cuda")
        ops.gemm_any(x, w, out=out[:M, :N])
        assert ((out[:M, :N] - z).abs() <= room).all()
        assert (out[M] == 7).all() and (out[:, N:] == 7).all()
        for i in range(M):   # (one row is gemm_any_rows_kernel's: the same sums in the same order, where its lanes take whole pieces)
            if K % 512 == 0:
                assert torch.equal(ops.gemm_any(x[i:i + 1], w), out[i:i + 1, :N])
        y = ops.gemm_any_act(x, w, bias=bias, act=_C.ACT_SIGMOID)
        assert ((y - torch.sigmoid(z + bias)).abs() <= room + 2.0 ** -21 * (1 + bias.abs())).all()
