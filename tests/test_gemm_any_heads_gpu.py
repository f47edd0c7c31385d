"""Per-head products of many rows (gemm_any_batched over bf16 weights) against fp64 over the rounded rows: row tiles' edges, every head depth
that has the kernel of its own and neighbours that have not, gates, strided columns, values that are not finite.

Bound: products of rounded operands are exact in fp32, the sum over K carries at most K roundings of 2^-24 of the absolute sum, the gate a
few more."""
import pytest
import torch

from nanovllm import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [65, 127, 128, 129, 511, 1027])
@pytest.mark.parametrize("H,N,K", [(16, 256, 128), (16, 128, 256), (3, 32, 64), (5, 512, 64), (2, 160, 128), (2, 96, 256), (2, 48, 128), (2, 128, 192)])
@pytest.mark.parametrize("gated", [False, True])
def test_heads(M, H, N, K, gated):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = (torch.randn(H, N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    x = torch.randn(M, H * (K + 8) + 16, device="cuda", generator=g)[:, 16:]     # heads K + 8 apart, columns of a wider buffer
    gate = torch.randn(M, H * N, device="cuda", generator=g) if gated else None
    full = torch.full((M + 1, H * (N + 4)), 7.0, device="cuda")
    ops.gemm_any_batched(x, K + 8, w, full[:M], N + 4, gate=gate, gate_batch=N)
    for h in range(H):
        xr = x[:, h * (K + 8):h * (K + 8) + K].bfloat16().double()
        want, size = xr @ w[h].double().T, xr.abs() @ w[h].double().abs().T
        if gated:
            want = want * torch.sigmoid(gate[:, h * N:(h + 1) * N].double())
        got = full[:M, h * (N + 4):h * (N + 4) + N].double()
        assert bool(((got - want).abs() <= (K + 16) * 2.0 ** -24 * size + 1e-6).all())
        assert bool((full[:M, h * (N + 4) + N:(h + 1) * (N + 4)] == 7.0).all())
    assert bool((full[M] == 7.0).all())


def test_rows_keep_to_themselves():
    """a row's result hangs on its own x row alone, whatever the others hold, and is the same in every tile"""
    g = torch.Generator(device="cuda").manual_seed(5)
    w = (torch.randn(4, 64, 128, device="cuda", generator=g) * 0.1).bfloat16()
    x = torch.randn(300, 4 * 128, device="cuda", generator=g)
    x[290] = x[7]
    a = torch.empty(300, 4 * 64, device="cuda")
    ops.gemm_any_batched(x, 128, w, a, 64)
    x[100], x[101] = float("nan"), float("inf")
    b = torch.empty_like(a)
    ops.gemm_any_batched(x, 128, w, b, 64)
    keep = [i for i in range(300) if i not in (100, 101)]
    assert torch.equal(a[290], a[7]) and torch.equal(a[keep], b[keep]) and bool(b[100].isnan().all())


def test_unaligned_columns():
    """columns that are no 16-byte pieces keep the general kernel"""
    g = torch.Generator(device="cuda").manual_seed(6)
    w = (torch.randn(3, 64, 64, device="cuda", generator=g) * 0.1).bfloat16()
    x = torch.randn(200, 3 * 64 + 1, device="cuda", generator=g)[:, 1:]
    out = torch.empty(200, 3 * 64, device="cuda")
    ops.gemm_any_batched(x, 64, w, out, 64)
    for h in range(3):
        want = x[:, h * 64:(h + 1) * 64].bfloat16().double() @ w[h].double().T
        assert (out[:, h * 64:(h + 1) * 64].double() - want).abs().max() <= 1e-4
