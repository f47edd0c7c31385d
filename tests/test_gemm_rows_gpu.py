"""The tile GEMM's small shapes (csrc/gemm_mid_kernel.hpp; 65 .. some hundred rows), its K slices, and the
sampler's candidates from logits in memory (csrc/gemm_pick.hip).

Tolerance: fp32 accumulation of K bf16 products (exact), K * 2^-24 of the sum of magnitudes, then the roundings to bf16 (2^-9 each; SwiGLU
rounds gate, silu(gate), up and the product)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from nanovllm import ops as o
    return o


def _operands(M, N, K):
    g = torch.Generator().manual_seed(M * 7 + N * 3 + K)
    x, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    return x.cuda(), w.cuda(), (x.float() @ w.float().T), (x.float().abs() @ w.float().abs().T)


@pytest.mark.parametrize("M", [1, 64, 65, 129, 200, 257])
@pytest.mark.parametrize("N,K", [(20, 64), (64, 128), (1000, 320), (1024, 3072), (4096, 1024)])
@pytest.mark.parametrize("bias", [False, True])
def test_rows_of_the_tile_gemm(ops, M, N, K, bias):
    x, w, want, mag = _operands(M, N, K)
    b = torch.linspace(-1, 1, N).bfloat16() if bias else None
    got = ops.gemm_tile(x, w, b.cuda() if bias else None).cpu().float()
    want = want + (b.float() if bias else 0)
    assert ((got - want).abs() <= (mag + 1) * K * 2.0 ** -24 + want.abs() * 2.0 ** -8 + 1e-30).all()


@pytest.mark.parametrize("M", [1, 65, 128, 200, 400])
@pytest.mark.parametrize("N,K", [(256, 64), (768, 192), (6144, 1024)])
def test_rows_of_the_swiglu_tile_gemm(ops, M, N, K):
    x, w, both, mag = _operands(M, N, K)
    gate, up = both[:, :N // 2], both[:, N // 2:]
    want = torch.nn.functional.silu(gate) * up
    got = ops.gemm_tile(x, w, silu_mul=True).cpu().float()
    slack = mag.max() * K * 2.0 ** -24 * 4
    assert ((got - want).abs() <= 2.0 ** -8 * (2 * want.abs() + (gate.abs() + 1) * up.abs()) + slack * (1 + up.abs() + gate.abs())).all()


@pytest.mark.parametrize("M", [1, 65, 200, 300])
@pytest.mark.parametrize("N,K,ks", [(20, 64, 1), (1024, 2048, 4), (1024, 3072, 4), (1000, 640, 2), (4096, 1024, 16)])
def test_rows_in_k_slices(ops, M, N, K, ks):
    x, w, want, mag = _operands(M, N, K)
    part = ops.gemm_tile_splitk(x, w, ks).cpu()
    assert part.shape == (ks, M, N)
    assert ((part.sum(0) - want).abs() <= (mag + 1) * (K + ks) * 2.0 ** -24 * 2).all()
    k = K // ks
    for s in range(ks):   # a slice's sum is that slice's
        own = x[:, s * k:(s + 1) * k].float() @ w[:, s * k:(s + 1) * k].float().T
        assert (part[s].cuda() - own).abs().max() <= 2.0 ** -24 * 2 * K * mag.max()


@pytest.mark.parametrize("M", [65, 130])
@pytest.mark.parametrize("N", [16, 8192, 8208, 20000])
def test_tokens_from_logits_in_memory(ops, M, N):
    """Greedy and sampled rows, equal logits (the first column wins): the tokens of argmax / sample over the same logits."""
    K = 64
    x, w, _, _ = _operands(M, N, K)
    packed = ops.pack_weight(w)
    temps = torch.linspace(0, 1.5, M).cuda()
    temps[::3] = 0
    rng = torch.tensor([1234, 9], dtype=torch.int64).cuda()
    out = torch.empty(M, dtype=torch.int64, device="cuda")
    x[1] = 0   # every logit equal
    logits, tokens = ops.gemm_packed_pick(x, packed, temps, rng, out, w=w)
    assert torch.equal(logits, ops.gemm_tile(x, w))
    assert torch.equal(tokens, ops.sample(logits, temps, 1234, 9))
    pairs = torch.empty((M, 2), dtype=torch.int32, device="cuda")
    ops.gemm_packed_pick(x, packed, None, rng, out, col_offset=1000, pairs_out=pairs, w=w)
    assert torch.equal(pairs[:, 1].long() - 1000, ops.argmax(logits))
    assert torch.equal(pairs[:, 0].contiguous().view(torch.float32), logits.float().max(1).values)
