"""The persistent head kernel over fp8 weights: logits against fp64 over the dequantised weights, the picks against the sampler over those logits,
at the edges of a chunk of rows and of the shapes that the kernel takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(16, 65536, 1024), (17, 65536, 1024), (32, 65568, 1024), (33, 65568, 1024), (63, 70016, 1024), (64, 65536, 1024),
                                   (65, 65536, 1024), (97, 65536, 1024), (130, 65536, 1024), (33, 65536, 896), (48, 65536, 896), (49, 65536, 896),
                                   (40, 65504, 1024)])
def test_head(M, N, K):
    from nanovllm import ops

    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = (torch.randn(M, K, device="cuda", generator=g) * 0.5).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).bfloat16()
    w[N - 1] = w[3]     # a tie between column 3 and the last one in every row
    packed = ops.pack_weight_fp8(w)
    q, scale = ops.quantize_fp8(w)
    wide = ops.dequantize_fp8(q, scale).double()
    plain = ops.gemm_packed(x, packed)
    want, size = x.double() @ wide.T, x.double().abs() @ wide.abs().T
    # fp32 sums of exact products in K steps, rounded to bf16 once
    assert bool(((plain.double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * size + 1e-6).all())
    temps = torch.zeros(M, device="cuda")
    temps[1::2] = torch.linspace(0.3, 1.7, M // 2, device="cuda")
    rng = torch.tensor([9, 77], dtype=torch.int64, device="cuda")
    logits, tokens = ops.gemm_packed_pick(x, packed, temps, rng, torch.full((M,), -1, dtype=torch.int64, device="cuda"))
    assert torch.equal(logits, plain) and torch.equal(tokens, ops.sample(plain, temps, seed=9, step=77))
    _, greedy = ops.gemm_packed_pick(x, packed, None, rng, torch.empty(M, dtype=torch.int64, device="cuda"))
    assert torch.equal(greedy, ops.argmax(plain))
