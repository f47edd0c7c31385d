"""True 32-bit products (gemm_any_f32_kernel) where a group's row tiles have workgroups of their own and where they are looked for, up to the largest number
of groups, and batches whose results do not lie on 16 bytes, against fp64.  Bound: exact products, at most K roundings of 2^-24 of the absolute sum, the
epilogue a handful more."""
import pytest
import torch

from nanovllm import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("counts,bound", [((9, 0, 33, 1), 40), ((32, 64, 65), 65), ((17,), 17), ((0, 0, 40, 0), 40), ((3,) * 200 + (70,), 70), ((1,) * 65534 + (40,), 40)])
def test_groups(counts, bound, dual):
    from nanovllm import ops

    G, P, N, K = len(counts), sum(counts), 33, 32
    g = torch.Generator(device="cuda").manual_seed(P)
    x = torch.randn(50, K, device="cuda", generator=g)
    rows = torch.randint(0, 50, (P,), device="cuda", generator=g, dtype=torch.int32)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    w, w2 = (torch.randn(G, N, K, device="cuda", generator=g) for _ in range(2))
    n = torch.tensor(counts)
    off = torch.cat([torch.zeros(1, dtype=torch.long), n.cumsum(0)]).int().cuda()
    y = ops.gemm_any_grouped_act(x, rows, w, w2 if dual else None, _C.ACT_SILU if dual else _C.ACT_NONE, off, bound, place, P)[place.long()].double()
    of = torch.repeat_interleave(torch.arange(G), n).cuda()
    xr = x[rows.long()].double().unsqueeze(1)
    step, ok = 8192, True
    for i in range(0, P, step):
        s = slice(i, i + step)
        a = w[of[s]].double()
        z, size = (xr[s] * a).sum(-1), (xr[s] * a).abs().sum(-1)
        if dual:
            b = w2[of[s]].double()
            z, size = torch.nn.functional.silu(z) * (xr[s] * b).sum(-1), 4 * size * ((xr[s] * b).abs().sum(-1) + 1)
        ok &= bool(((y[s] - z).abs() <= (K + 16) * 2.0 ** -24 * size + 1e-6).all())
    assert ok


@pytest.mark.parametrize("M,N,shift", [(70, 36, 0), (100, 33, 1), (65, 64, 2)])
def test_batches_off_16_bytes(M, N, shift):
    """each batch's rows of the result begin where they begin, whatever the first one's do"""
    from nanovllm import ops

    B, K = 3, 64
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = torch.randn(M, B * K, device="cuda", generator=g), torch.randn(B, N, K, device="cuda", generator=g)
    out = torch.full((M, 4 * (B * (N + shift) // 4 + 2)), 7.0, device="cuda")
    ops.gemm_any_batched(x, K, w, out, N + shift)
    for b in range(B):
        xr = x[:, b * K:(b + 1) * K].double()
        got = out[:, b * (N + shift):b * (N + shift) + N].double()
        assert bool(((got - xr @ w[b].double().T).abs() <= (K + 16) * 2.0 ** -24 * (xr.abs() @ w[b].double().abs().T)).all())
        assert bool((out[:, b * (N + shift) + N:(b + 1) * (N + shift)] == 7.0).all())
