"""fp32-activation products of up to eight rows, one and four features per wave (csrc/gemm_any.hip: gemm_any_rows_kernel), a soft-capped
product on the tile kernels, and the grouped router's picks (csrc/seqmix.hip) at the borders of a lane's outputs.

Tolerance of the products: lane sums of K / 64 fp32 terms and a butterfly of six additions, each 2^-24 of the sum of magnitudes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from nanovllm import ops as o
    return o


@pytest.mark.parametrize("M", [1, 3, 4, 8])
@pytest.mark.parametrize("K", [8, 100, 520, 2048])
@pytest.mark.parametrize("N", [8192, 8195])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("odd", [False, True])
def test_rows_with_one_and_four_features_per_wave(ops, M, K, N, dtype, odd):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K + odd, device="cuda", generator=g)[:, odd:]   # odd: rows off 16 bytes
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(dtype)
    got = ops.gemm_any(x, w)
    want = x.double() @ w.double().T
    mag = x.double().abs() @ w.double().abs().T
    assert ((got.double() - want).abs() <= (K / 64 + 16) * 2.0 ** -24 * mag + 1e-12).all()
    few = ops.gemm_any(x, w[-60:].contiguous())   # fewer features: one per wave, the same order of sums
    assert torch.equal(got[:, -60:], few)


@pytest.mark.parametrize("M,N,K", [(9, 8192, 64), (24, 100, 512), (200, 260, 128)])
def test_soft_capped_rows_on_the_tile_kernels(ops, M, N, K):
    from nanovllm import _C
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, w = torch.randn(M, K, device="cuda", generator=g) * 3, (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    assert ops._tile_rows(M, w, None, _C.ACT_SOFTCAP, False, 0) == 64
    z = x.bfloat16().double() @ w.double().T
    mag = x.bfloat16().double().abs() @ w.double().abs().T
    got = ops.gemm_any_act(x, w, act=_C.ACT_SOFTCAP, alpha=5.0)
    assert ((got.double() - 5 * torch.tanh(z / 5)).abs() <= (K + 16) * 2.0 ** -24 * mag + 5 * 2.0 ** -21).all()


@pytest.mark.parametrize("n,groups,keep,top", [(3, 1, 1, 3), (64, 4, 2, 8), (65, 5, 3, 7), (128, 8, 8, 8), (200, 10, 4, 6), (512, 16, 2, 16)])
def test_grouped_picks(ops, n, groups, keep, top):
    """Scores with many ties (the lower output first), zeros of both signs, a NaN logit (counts as score 0)."""
    g = torch.Generator().manual_seed(n)
    T = 9
    z = torch.randint(-3, 4, (T, n), generator=g).float()
    corr = torch.randint(-1, 2, (n,), generator=g).float() * 0.0 + torch.where(torch.arange(n) % 7 == 3, -0.0, 0.0)
    z[4, n // 2] = float("nan")
    from nanovllm import _C
    ids, wts = ops.route_grouped(z.cuda(), corr.cuda(), top, groups, keep, _C.ROUTE_SIGMOID, _C.ROUTE_GROUP_MAX)
    score = torch.sigmoid(z)
    score[score.isnan()] = 0.0
    for t in range(T):
        s = score[t] + corr + 0.0
        best = s.view(groups, -1).max(1).values
        kept = sorted(range(groups), key=lambda i: (-best[i].item(), i))[:keep]
        per = n // groups
        allowed = [e for e in range(n) if e // per in kept]
        want = sorted(allowed, key=lambda e: (-s[e].item(), e))[:top]
        assert ids[t].tolist() == want
        assert (wts[t].cpu() - score[t][want]).abs().max() <= 2.0 ** -22


@pytest.mark.parametrize("counts", [(1, 0, 1, 1, 0, 0, 0, 1), (0, 4, 0, 0), (1,) * 8, (0, 0, 0, 0, 0, 0, 0, 8), (0, 11, 1) + (0,) * 11])
@pytest.mark.parametrize("K", [8, 100, 1032])
@pytest.mark.parametrize("dtype,exact", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float32, False)])
@pytest.mark.parametrize("dual", [False, True])
def test_groups_of_a_row_or_none(ops, counts, K, dtype, exact, dual):
    """no more rows than groups: one row after the other (gemm_any_each_row_kernel); the order of sums is a plain product's of a row"""
    G, N, P = len(counts), 21, sum(counts)
    g = torch.Generator(device="cuda").manual_seed(K + P)
    x = torch.randn(5, K, device="cuda", generator=g)
    rows = torch.randint(0, 5, (P,), device="cuda", generator=g, dtype=torch.int32)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    w, w2 = ((torch.randn(G, N, K, device="cuda", generator=g) * K ** -0.5).to(dtype) for _ in range(2))
    got = ops.gemm_any_grouped(x, rows, w, w2 if dual else None, off, P, place, P, exact)
    for e in range(G):
        for m in range(int(off[e]), int(off[e + 1])):
            one = x[rows[m].long()][None]
            if P > 8 and not exact:   # (only then is x rounded, and not here)
                continue
            z = ops.gemm_any(one, w[e], exact=True)[0]
            if dual:
                z = torch.nn.functional.silu(z.double()) * ops.gemm_any(one, w2[e], exact=True)[0].double()
                assert ((got[place[m].long()].double() - z).abs() <= 2.0 ** -20 * z.abs() + 1e-12).all()
            else:
                assert torch.equal(got[place[m].long()], z)


@pytest.mark.parametrize("M", [2, 3, 5, 6, 7, 8, 9, 11, 13, 64])
@pytest.mark.parametrize("K", [8, 520, 1000, 1024])
@pytest.mark.parametrize("N", [33, 4100])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dual", [False, True])
def test_batches_of_every_size(ops, M, K, N, dtype, dual):
    """every row has the bits that it has alone, whatever its batch and however many pieces of K are asked for together"""
    from nanovllm import _C
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K, device="cuda", generator=g)
    w, w2 = ((torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(dtype) for _ in range(2))
    kw = dict(act=_C.ACT_SILU, w2=w2) if dual else {}
    got = ops.gemm_any_act(x, w, exact=True, **kw)
    one = torch.cat([ops.gemm_any_act(x[r:r + 1], w, exact=True, **kw) for r in range(M)])
    assert torch.equal(got, one)
    z, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bound = (K / 64 + 16) * 2.0 ** -24 * mag + 1e-12
    if dual:   # (silu is 1.1-Lipschitz and at most its argument)
        z2, mag2 = x.double() @ w2.double().T, x.double().abs() @ w2.double().abs().T
        bound = 1.1 * bound * (z2.abs() + (K / 64 + 16) * 2.0 ** -24 * mag2) + z.abs() * (K / 64 + 16) * 2.0 ** -24 * mag2 + 2.0 ** -20 * (z * z2).abs() + 1e-12
        z = torch.nn.functional.silu(z) * z2
    assert ((got.double() - z).abs() <= bound).all()


@pytest.mark.parametrize("counts", [(8,), (3, 5), (0, 7, 1), (5, 0, 12, 4), (33, 31)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_groups_in_batches_of_four(ops, counts, dtype):
    G, N, K, P = len(counts), 37, 600, sum(counts)
    g = torch.Generator(device="cuda").manual_seed(P)
    x = torch.randn(P, K, device="cuda", generator=g)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    w = (torch.randn(G, N, K, device="cuda", generator=g) * K ** -0.5).to(dtype)
    got = ops.gemm_any_grouped(x, None, w, None, off, P, None, P, True)
    for e in range(G):
        for m in range(int(off[e]), int(off[e + 1])):
            assert torch.equal(got[m], ops.gemm_any(x[m:m + 1], w[e], exact=True)[0])
