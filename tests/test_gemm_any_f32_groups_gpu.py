"""True 32-bit grouped products (gemm_any_f32_kernel over the row tiles of all groups) against fp64: more groups than a wave has lanes, empty and
one-row groups, more row tiles than the launch has workgroups for, one and two weights, rows scattered on both sides.

Bound: exact products, at most K roundings of 2^-24 of the absolute sum, the epilogue a handful more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("G,P,bound,N,K", [(5, 700, None, 96, 64), (70, 1500, None, 64, 32), (130, 900, None, 40, 96), (8, 4000, 600, 1030, 32),
                                           (3, 9000, 3500, 68, 32), (33, 2912, None, 512, 256), (2, 40, None, 32, 64)])
def test_groups(G, P, bound, N, K, dual):
    from nanovllm import _C, ops

    g = torch.Generator(device="cuda").manual_seed(G + P)
    share = torch.rand(G, generator=torch.Generator().manual_seed(P)) + 0.05
    share[::4] = 0
    if bound:
        share[:] = 1.0
    counts = (share / share.sum() * (P - 10)).long().tolist()
    counts[-1] = max(counts[-1], 1)
    if not bound and G > 4:
        counts[1] = 1
    assert not bound or max(counts) <= bound
    total = sum(counts)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    T = P // 3
    x = torch.randn(T, K, device="cuda", generator=g)
    rows = torch.randint(0, T, (P,), device="cuda", generator=g, dtype=torch.int32)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    w, w2 = (torch.randn(G, N, K, device="cuda", generator=g) * K ** -0.5 for _ in range(2))
    act = _C.ACT_SILU if dual else _C.ACT_NONE
    y = ops.gemm_any_grouped_act(x, rows, w, w2 if dual else None, act, off, bound or P, place, P)
    for e, n in enumerate(counts):
        r = slice(int(off[e]), int(off[e]) + n)
        xr, at = x[rows[r].long()].double(), place[r].long()
        z, size = xr @ w[e].double().T, xr.abs() @ w[e].double().abs().T
        if dual:
            z2, s2 = xr @ w2[e].double().T, xr.abs() @ w2[e].double().abs().T
            z, size = torch.nn.functional.silu(z) * z2, 4 * size * (s2 + 1)
        assert bool(((y[at].double() - z).abs() <= (K + 16) * 2.0 ** -24 * size + 1e-6).all()), e
    assert total > 8
