"""gemm_any_split_kernel: 32-bit products as three bf16 parts of each operand, at the edges of its tiles, rings and groups, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from nanovllm import ops
    return ops


def _bound(x, w, K):
    """products left out: 2^-25 of |x w|; sums: K roundings at most, of either sum"""
    return (K + 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -140


# 64 x 64 and 128 x 64 tiles, part-filled in both directions; K loops of 1 .. 5 steps and longer ones
@pytest.mark.parametrize("M,N,K", [(16384, 4100, 32), (8193, 4100, 64), (4097, 4100, 96), (4096, 4100, 128), (4095, 4099, 160),
                                   (721, 3072, 1024), (1999, 1101, 1024), (4001, 2050, 544)])
def test_split_products(ops, M, N, K):
    g = torch.Generator().manual_seed(M + K)
    buf = torch.randn(M, K + 4, generator=g).to(DEV)
    x, w = buf[:, :K], torch.randn(N, K, generator=g).to(DEV)
    out = torch.full((M + 1, N), 7.0, device=DEV)
    y = ops.gemm_any(x, w, exact=True, out=out[:M])
    rows = torch.cat([torch.arange(0, 130), torch.arange(M - 130, M)]).to(DEV)
    want = x[rows].double() @ w.double().T
    assert bool(((y[rows].double() - want).abs() <= _bound(x[rows], w, K)).all())
    assert bool((out[M] == 7.0).all())


@pytest.mark.parametrize("E,pairs,N,K", [(7, 6000, 512, 1024), (32, 2884, 500, 1024), (5, 4000, 1030, 512)])
def test_split_products_of_groups(ops, E, pairs, N, K):
    """ragged groups, empty ones and one of a single row among them; one weight and two"""
    g = torch.Generator().manual_seed(E)
    share = torch.rand(E, generator=g) + 0.2
    share[E // 2] = 0.0
    count = (share / share.sum() * (pairs - 1)).int()
    count[0] += pairs - 1 - int(count.sum())
    count[E - 1] += 1
    count[E // 2 - 1], count[0] = 1, count[0] + count[E // 2 - 1] - 1
    off = torch.zeros(E + 1, dtype=torch.int32)
    off[1:] = count.cumsum(0)
    assert int(off[E]) == pairs
    x = torch.randn(pairs // 3, K, generator=g).to(DEV)
    xr = torch.randint(0, pairs // 3, (pairs,), generator=g).to(torch.int32).to(DEV)
    yr = torch.randperm(pairs, generator=g).to(torch.int32).to(DEV)
    w, w2 = (torch.randn(E, N, K, generator=g).to(DEV) * K ** -0.5 for _ in range(2))
    one = ops.gemm_any_grouped(x, xr, w, None, off.to(DEV), pairs, yr, pairs, exact=True)
    two = ops.gemm_any_grouped(x, xr, w, w2, off.to(DEV), pairs, yr, pairs, exact=True)
    for e in range(E):
        r = slice(int(off[e]), int(off[e + 1]))
        if r.start == r.stop:
            continue
        xe, at = x[xr[r].long()], yr[r].long()
        z, u = xe.double() @ w[e].double().T, xe.double() @ w2[e].double().T
        bz, bu = _bound(xe, w[e], K), _bound(xe, w2[e], K)
        assert bool(((one[at].double() - z).abs() <= bz).all()), e
        want = torch.nn.functional.silu(z) * u
        # silu's slope is at most 1.1; its own arithmetic and the product: a few roundings of the value
        assert bool(((two[at].double() - want).abs() <= 1.1 * bz * u.abs() + (torch.nn.functional.silu(z).abs() + 1.1 * bz) * bu + 2.0 ** -20 * want.abs()).all()), e


def test_split_products_of_numbers_without_parts(ops):
    """infinities, NaN, numbers next to the largest and far below the smallest whose parts bf16 holds"""
    M, N, K = 2000, 1100, 1024
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    x[3, 5], x[70, 9], w[11, 2], x[1999, 1023] = float("inf"), float("nan"), float("-inf"), float("-inf")
    x[40] *= 2.0 ** -118
    x[41, 1], w[:, 1] = 3.4e38, 0.25
    x[42] = 0.0
    y = ops.gemm_any(x.to(DEV), w.to(DEV), exact=True).cpu()
    want = x.double() @ w.double().T
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isposinf(), want.isposinf()) and torch.equal(y.isneginf(), want.isneginf())
    fine = want.isfinite()
    xs, ws = torch.where(x.isfinite(), x, 0.0), torch.where(w.isfinite(), w, 0.0)
    err = torch.where(fine, (y.double() - want).abs(), torch.zeros((), dtype=torch.float64))
    assert bool((err <= torch.where(fine, _bound(xs, ws, K), 1.0)).all())
    tiny = want[40, 12:]
    assert float((y[40, 12:].double() - tiny).norm() / tiny.norm()) <= K * 2.0 ** -24
    assert bool((y[42, 12:] == 0).all())


# x of 2^a, weights of 2^b: operands below what three bf16 parts hold, against large ones (outputs that are ordinary numbers), either way round
@pytest.mark.parametrize("a,b", [(-116, 36), (-120, 79), (-124, 40), (-130, 60), (-138, 79), (36, -116), (60, -130), (-60, -60)])
def test_split_products_of_small_operands(ops, a, b):
    M, N, K = 2000, 1100, 1024
    g = torch.Generator().manual_seed(5 - a)
    x, w = (torch.randn(M, K, generator=g) * 2.0 ** a).to(DEV), (torch.randn(N, K, generator=g) * 2.0 ** b).to(DEV)
    y = ops.gemm_any(x, w, exact=True)
    want = x.double() @ w.double().T
    # as of ordinary operands: 2^-24 a rounding; a bf16 part less is 3.5e-6
    assert float((y.double() - want).norm() / want.norm()) <= 4e-7


# rows that have no finite parts (NaN, infinities, numbers from 2^104 on) in a batch: every other row's bits, those 16 rows on among them, are its own, and
# a row whose outputs are finite all the same has the fp32 kernel's accuracy
@pytest.mark.parametrize("dual", [False, True])
def test_split_products_rows_keep_their_bits(ops, dual):
    from nanovllm import _C

    M, N, K = 2049, 2050, 1024
    g = torch.Generator().manual_seed(11)
    x, w, w2 = (torch.randn(n, K, generator=g).to(DEV) for n in (M, N, N))
    product = lambda rows: ops.gemm_any_act(rows, w, act=_C.ACT_SILU if dual else _C.ACT_NONE, w2=w2 if dual else None, exact=True)
    want = product(x)
    odd = x.clone()
    bad = {5: float("nan"), 70: float("inf"), 83: 2.0 ** 105, 1000: 3.4e38, 2032: float("-inf"), 2048: 2.0 ** 120}
    for r, v in bad.items():
        odd[r, r % K] = v
    odd[86] *= 2.0 ** 100   # (sums beyond 2^80)
    got = product(odd)
    same = torch.ones(M, dtype=torch.bool, device=DEV)
    same[list(bad) + [86]] = False
    assert torch.equal(got[same].view(torch.int32), want[same].view(torch.int32))
    if not dual:
        big = odd[[83, 86]].double() @ w.double().T
        assert bool(((got[[83, 86]].double() - big).abs() <= _bound(odd[[83, 86]], w, K)).all())
    assert bool(got[5].isnan().all()) and not bool(got[70].isfinite().any())


def test_split_products_of_single_terms(ops):
    """sums of one nonzero product, which fp32 arithmetic rounds once: what is left out (l l, below 2^-34 of it) and the rounding of the low sum (below
    2^-31) are some 0.01 of a last bit"""
    M, N, K = 2049, 2050, 1024
    g = torch.Generator().manual_seed(17)
    at = torch.randint(0, K, (M,), generator=g).to(DEV)
    x, w, v = torch.zeros(M, K, device=DEV), torch.randn(N, K, generator=g).to(DEV), torch.randn(M, generator=g).to(DEV)
    x[torch.arange(M, device=DEV), at] = v
    want = v.double()[:, None] * w.double().T[at]
    ulp = torch.exp2(torch.floor(torch.log2(want.abs())) - 23)
    assert float(((ops.gemm_any(x, w, exact=True).double() - want).abs() / ulp).max()) <= 0.52
