"""The exact (true 32-bit) products of the 32-bit-residual families on the fp32 matrix instruction: edges of the three tiles, fp32
and bf16 weights, gathered and scattered groups, against float64.  Bound: a sum of K products in any order carries at most K
roundings of 2^-24 of the absolute sum, the epilogue a few more."""
import pytest
import torch

from nanovllm import _C, ops

pytestmark = pytest.mark.gpu


def _close(got, want, size, K):
    err = (got.double() - want).abs()
    bound = (K + 16) * 2.0 ** -24 * size + 1e-7
    assert bool((err <= bound).all()), float((err / bound).max())
    assert float((err.pow(2).sum() / want.pow(2).sum()).sqrt()) < 2e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(65, 1, 32), (65, 33, 64), (97, 64, 96), (130, 65, 128), (733, 136, 256), (1100, 1027, 160), (70, 40, 48),
                                   (66, 40, 30)])
def test_plain_rows(dtype, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 4, device="cuda", generator=g)[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g).mul(K ** -0.5).to(dtype)
    bias = torch.randn(N, device="cuda", generator=g)
    out = torch.full((M + 1, N), 7.0, device="cuda")
    ops.gemm_any_act(x, w, bias=bias, alpha=0.5, exact=True, out=out[:M])
    want = 0.5 * (x.double() @ w.double().T + bias)
    _close(out[:M], want, x.double().abs() @ w.double().abs().T + bias.abs(), K)
    assert bool((out[M] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("counts", [(100, 0, 1, 64, 65), (33, 32, 0), (200, 3)])
@pytest.mark.parametrize("dual", [False, True])
def test_grouped_rows(dtype, counts, dual):
    G, N, K, T = len(counts), 72, 96, 50
    P = sum(counts)
    g = torch.Generator(device="cuda").manual_seed(P + dual)
    x = torch.randn(T, K, device="cuda", generator=g)
    rows = torch.randint(0, T, (P,), device="cuda", generator=g, dtype=torch.int32)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    w, w2 = (torch.randn(G, N, K, device="cuda", generator=g).mul(K ** -0.5).to(dtype) for _ in range(2))
    y = ops.gemm_any_grouped_act(x, rows, w, w2 if dual else None, _C.ACT_SILU if dual else _C.ACT_NONE, off, P, place, P, exact=True)
    want, size = torch.zeros(P, N, device="cuda", dtype=torch.float64), torch.ones(P, N, device="cuda", dtype=torch.float64)
    for e in range(G):
        r = slice(int(off[e]), int(off[e + 1]))
        xr, at = x[rows[r].long()].double(), place[r].long()
        z = xr @ w[e].double().T
        s = xr.abs() @ w[e].double().abs().T
        want[at] = torch.nn.functional.silu(z) * (xr @ w2[e].double().T) if dual else z
        size[at] = 3 * s * (xr.abs() @ w2[e].double().abs().T + 1) if dual else s
    _close(y, want, size, K)


def test_a_row_has_the_same_bits_in_every_tile():
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(5000, 256, device="cuda", generator=g), torch.randn(96, 256, device="cuda", generator=g)
    whole = ops.gemm_any(x, w, exact=True)
    assert torch.equal(whole[:700], ops.gemm_any(x[:700], w, exact=True)) and torch.equal(whole[17:90], ops.gemm_any(x[17:90], w, exact=True))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,odd", [(1024, 64, 40, 0), (1039, 5, 100, 0), (1500, 33, 64, 1), (1023, 64, 40, 0), (1024, 65, 40, 0)])
def test_few_features_over_rows_that_are_no_whole_lines(dtype, M, N, K, odd):
    """16-row tiles up to 64 features and from 1024 rows on, 64-row tiles beside that; the bound as above"""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + odd, device="cuda", generator=g)[:, odd:]
    w = torch.randn(N, K, device="cuda", generator=g).to(dtype)
    got, want = ops.gemm_any(x, w, exact=True), x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    assert bool(((got.double() - want).abs() <= K * 2.0 ** -23 * size + 1e-12).all())


@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192])
@pytest.mark.parametrize("M,N,dtype,dual", [(130, 40, torch.float32, False), (300, 200, torch.float32, True), (700, 512, torch.bfloat16, False),
                                            (1300, 900, torch.float32, False), (1300, 900, torch.bfloat16, True), (400, 1408, torch.bfloat16, True)])
def test_fragments_read_a_step_ahead(M, N, dtype, dual, K):
    """one to six K steps (fewer than the ring holds, odd and even) of every tile size: K roundings of the terms' sum"""
    from nanovllm import _C, ops
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn(M, K, device="cuda", generator=g)
    w, w2 = (torch.randn(N, K, device="cuda", generator=g).to(dtype) for _ in range(2))
    got = ops.gemm_any_act(x, w, None, _C.ACT_SILU, w2=w2, exact=True) if dual else ops.gemm_any(x, w, exact=True)
    z, size = x.double() @ w.double().T, x.abs().double() @ w.abs().double().T
    tol = (K + 4) * 2.0 ** -24 * size
    if dual:   # |silu'| < 1.1, |silu(z)| <= |z|; its own form adds a few roundings of the result
        u, usize = x.double() @ w2.double().T, x.abs().double() @ w2.abs().double().T
        want = torch.nn.functional.silu(z) * u
        tol = 1.1 * tol * u.abs() + z.abs() * (K + 4) * 2.0 ** -24 * usize + 16 * 2.0 ** -24 * want.abs() + tol * (K + 4) * 2.0 ** -24 * usize
    else:
        want = z
    assert bool(((got.double() - want).abs() <= tol).all())

