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
    """products left out: 2^-34 of |x w|; sums: K roundings at most, of either sum"""
    return (K + 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -140


def _close(y, want, K, factors=1):
    """The kernel's own accuracy (2-norm): a rounding of either sum per 32 of K, some 6e-9 sqrt(K) and a last one.  A part less in the operands is 3.5e-6;
    the fp32 matrix instruction, with eight roundings per 32 of K, has 1.8e-8 sqrt(K) and fails too: these launches run on the kernel.  factors: two
    for the product of two sums."""
    err = float((y.double() - want).norm() / want.norm())
    assert err <= (2.5e-8 + 9e-9 * K ** 0.5) * factors ** 0.5, err


# tiles part-filled in both directions; K loops of 1 .. 5 steps and longer ones; rows whose stride is no whole line
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
    _close(y[rows], want, K)
    assert bool((out[M] == 7.0).all())
    # (a row's bits do not depend on its place)
    assert torch.equal(ops.gemm_any(x[1:], w, exact=True).view(torch.int32), y[1:].view(torch.int32))


@pytest.mark.parametrize("E,pairs,N,K", [(7, 12000, 512, 1024), (32, 12000, 500, 1024), (130, 20000, 257, 512), (1, 9000, 700, 512)])
def test_split_products_of_groups(ops, E, pairs, N, K):
    """two weights of ragged groups, empty ones and one of a single row among them"""
    g = torch.Generator().manual_seed(E)
    share = torch.rand(E, generator=g) + 0.2
    if E > 1:
        share[E // 2] = 0.0
    count = (share / share.sum() * (pairs - 1)).int()
    count[0] += pairs - int(count.sum())
    if E > 1:
        count[0] += count[E // 2 - 1] - 1
        count[E // 2 - 1] = 1
    off = torch.zeros(E + 1, dtype=torch.int32)
    off[1:] = count.cumsum(0)
    assert int(off[E]) == pairs
    x = torch.randn(pairs // 3, K, generator=g).to(DEV)
    xr = torch.randint(0, pairs // 3, (pairs,), generator=g).to(torch.int32).to(DEV)
    yr = torch.randperm(pairs, generator=g).to(torch.int32).to(DEV)
    w, w2 = (torch.randn(E, N, K, generator=g).to(DEV) * K ** -0.5 for _ in range(2))
    two = ops.gemm_any_grouped(x, xr, w, w2, off.to(DEV), pairs, yr, pairs, exact=True)
    for e in range(E):
        r = slice(int(off[e]), int(off[e + 1]))
        if r.start == r.stop:
            continue
        xe, at = x[xr[r].long()], yr[r].long()
        z, u = xe.double() @ w[e].double().T, xe.double() @ w2[e].double().T
        bz, bu = _bound(xe, w[e], K), _bound(xe, w2[e], K)
        want = torch.nn.functional.silu(z) * u
        # silu's slope is at most 1.1; its own arithmetic and the product: a few roundings of the value
        assert bool(((two[at].double() - want).abs() <= 1.1 * bz * u.abs() + (torch.nn.functional.silu(z).abs() + 1.1 * bz) * bu + 2.0 ** -20 * want.abs()).all()), e
        if r.stop - r.start > 16:
            _close(two[at], want, K, factors=3)   # (two sums, silu's and the product's roundings)


@pytest.mark.parametrize("M,N,K,pad", [(2049, 2050, 1024, 0), (3000, 1500, 768, 3)])
def test_split_products_of_two_weights(ops, M, N, K, pad):
    from nanovllm import _C

    g = torch.Generator().manual_seed(N)
    x, w, w2 = (torch.randn(n, K, generator=g).to(DEV) * s for n, s in ((M, 1.0), (N, K ** -0.5), (N, K ** -0.5)))
    b, b2 = (torch.randn(N, generator=g).to(DEV) for _ in range(2))
    out = torch.full((M + 1, N + pad), 7.0, device=DEV)   # (pad 3: single stores)
    y = ops.gemm_any_act(x, w, bias=b, act=_C.ACT_SILU, w2=w2, bias2=b2, alpha=0.5, exact=True, out=out[:M, :N])
    want = 0.5 * torch.nn.functional.silu(x.double() @ w.double().T + b) * (x.double() @ w2.double().T + b2)
    _close(y, want, K, factors=3)
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


def test_split_products_with_epilogues(ops):
    from nanovllm import _C

    M, N, K = 2049, 2050, 1024
    g = torch.Generator().manual_seed(3)
    x, w, b = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV) * K ** -0.5, torch.randn(N, generator=g).to(DEV)
    z = x.double() @ w.double().T + b
    _close(ops.gemm_any_act(x, w, bias=b, alpha=3.0, exact=True), 3.0 * z, K, factors=2)
    _close(ops.gemm_any_act(x, w, bias=b, act=_C.ACT_RELU2, exact=True), z.clamp(min=0) ** 2, K, factors=8)
    # a segment without an activation, one with each of two
    y = ops.gemm_any_segments(x, w, b, _C.ACT_SIGMOID, 700, _C.ACT_TANH, 1501, exact=True)
    _close(y[:, :700], z[:, :700], K, factors=2)
    # (slopes of at most 1; the functions' own arithmetic: a few roundings)
    assert float((y[:, 700:1501].double() - z[:, 700:1501].sigmoid()).abs().max()) <= 2e-6
    assert float((y[:, 1501:].double() - z[:, 1501:].tanh()).abs().max()) <= 3e-6


@pytest.mark.parametrize("gated", [False, True])
def test_split_products_of_batches(ops, gated):
    B, M, N, K = 16, 2049, 500, 512
    g = torch.Generator().manual_seed(B + gated)
    x, w = torch.randn(M, B * K + 8, generator=g).to(DEV), torch.randn(B, N, K, generator=g).to(DEV) * K ** -0.5
    gate = torch.randn(M, B * 504, generator=g).to(DEV) if gated else None
    out = torch.full((M, B * 504), 7.0, device=DEV)
    ops.gemm_any_batched(x, K, w, out, 504, gate=gate, gate_batch=504, exact=True)
    for h in range(B):
        want = x[:, h * K:(h + 1) * K].double() @ w[h].double().T
        if gated:
            want *= gate[:, h * 504:h * 504 + N].double().sigmoid()
        _close(out[:, h * 504:h * 504 + N], want, K, factors=3 if gated else 1)
    assert bool((out.view(M, B, 504)[:, :, N:] == 7.0).all())


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
    assert float((y.double() - want).norm() / want.norm()) <= 3.2e-7


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
