"""Products of decode batches and of experts of a few rows each (csrc/gemm_any.hip: gemm_any_stream_kernel) against float64 over the
rounded operands.

Bound: the operands' products are exact in fp32; the sum over K carries at most K roundings of 2^-24 of the absolute sum, the epilogue
a handful more; silu is 1.1-Lipschitz and at most its argument, sigmoid and tanh 1-Lipschitz."""
import pytest
import torch

from nanovllm import _C

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from nanovllm import ops as o
    return o


def _make(M, N, K, seed, batch=None):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K + 8, device="cuda", generator=g)[:, 4:4 + K]   # rows on 16 bytes inside wider ones
    w, w2 = ((torch.randn(*([batch] if batch else []), N, K, device="cuda", generator=g) * K ** -0.5).bfloat16() for _ in range(2))
    return g, x, w, w2


def _ok(got, want, mag, K):
    err = (got.double() - want).abs()
    bound = (K + 16) * 2.0 ** -24 * mag + 1e-6
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("M", [9, 16, 17, 31, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(1, 64), (17, 128), (100, 1088), (2052, 576), (6145, 192), (16384, 64)])
def test_plain(ops, M, N, K):
    g, x, w, w2 = _make(M, N, K, M + N + K)
    assert _C.lib.mi_gemm_any_streams(M, N, K, 0) == (M <= 32 or N <= (6144 if M <= 48 else 4096))
    xr, bias = x.bfloat16().double(), torch.randn(N, device="cuda", generator=g)
    z, mag = xr @ w.double().T, xr.abs() @ w.double().abs().T
    out = torch.full((M + 1, N + 3), 7.0, device="cuda")
    ops.gemm_any(x, w, alpha=0.5, out=out[:M, :N])   # (rows of the result off 16 bytes where N says so)
    _ok(out[:M, :N], 0.5 * z, mag, K)
    assert bool((out[M] == 7.0).all() and (out[:, N:] == 7.0).all())
    _ok(ops.gemm_any_act(x, w, bias=bias, act=_C.ACT_SIGMOID), torch.sigmoid(z + bias), mag + bias.abs(), K)
    _ok(ops.gemm_any_act(x, w, act=_C.ACT_SOFTCAP, alpha=5.0), 5 * torch.tanh(z / 5), mag + 1, K)
    if N <= 2052:
        z2, m2 = xr @ w2.double().T, xr.abs() @ w2.double().abs().T
        _ok(ops.gemm_any_act(x, w, act=_C.ACT_SILU, w2=w2), torch.nn.functional.silu(z) * z2, 3 * mag * (m2 + 1), K)
        at = N // 3
        want = torch.cat([z[:, :at], torch.tanh(z[:, at:])], 1)
        _ok(ops.gemm_any_segments(x, w, None, _C.ACT_TANH, at), want, mag + 1, K)


def test_a_row_depends_on_itself_alone(ops):
    """whatever the batch: rows of 9, 16 and 30 have the bits they have among 64 fewer or more, and NaN and infinities stay in theirs"""
    _, x, w, _ = _make(32, 300, 640, 5)
    x = x.clone()
    x[3, 7], x[20, 600] = float("nan"), float("inf")
    y = ops.gemm_any(x, w)
    clean = [r for r in range(32) if r not in (3, 20)]
    assert bool(y[clean].isfinite().all()) and bool(y[3].isnan().all()) and not bool(y[20].isfinite().any())
    for n in (17, 25):
        assert torch.equal(ops.gemm_any(x[:n], w)[4:17], y[4:17])


@pytest.mark.parametrize("M", [9, 24, 40, 64])
@pytest.mark.parametrize("H,N,K", [(3, 130, 128), (8, 64, 256)])
def test_batches(ops, M, H, N, K):
    g, _, w, _ = _make(1, N, K, M + N, H)
    x = torch.randn(M, H * K, device="cuda", generator=g)
    gate = torch.randn(M, H * N, device="cuda", generator=g)
    out = torch.empty(M, H * N, device="cuda")
    ops.gemm_any_batched(x, K, w, out, N, gate=gate, gate_batch=N)
    for h in range(H):
        xr, s = x[:, h * K:(h + 1) * K].bfloat16().double(), slice(h * N, (h + 1) * N)
        _ok(out[:, s], xr @ w[h].double().T * torch.sigmoid(gate[:, s].double()), xr.abs() @ w[h].double().abs().T, K)


@pytest.mark.parametrize("counts", [(3, 0, 16, 1, 17, 2, 0, 9), (33,) + (0,) * 7, (1,) * 16, (70, 0, 5) + (1,) * 9])
@pytest.mark.parametrize("K,N", [(64, 20), (320, 2052)])
def test_groups(ops, counts, K, N):
    G, P, T = len(counts), sum(counts), 13
    g, x, w, w2 = _make(T, N, K, P + N, G)
    rows = torch.randint(0, T, (P,), device="cuda", generator=g, dtype=torch.int32)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    scale = torch.rand(P, device="cuda", generator=g)
    assert P > 8 and _C.lib.mi_gemm_any_streams(P, N, K, G)
    one = ops.gemm_any_grouped(x, rows, w, None, off, P, place, P)
    two = ops.gemm_any_grouped_glu(x, rows, w, w2, _C.ACT_CLAMPED_GLU, 1.5, scale, place, off, P, place, P)
    for e in range(G):
        r = slice(int(off[e]), int(off[e + 1]))
        xr, at = x[rows[r].long()].bfloat16().double(), place[r].long()
        z, z2 = xr @ w[e].double().T, xr @ w2[e].double().T
        m, m2 = xr.abs() @ w[e].double().abs().T, xr.abs() @ w2[e].double().abs().T
        _ok(one[at], z, m, K)
        f = scale[at].double().unsqueeze(1)
        c, u = (z * f).clamp(max=1.5), (z2 * f).clamp(-1.5, 1.5)
        _ok(two[at], c * torch.sigmoid(1.702 * c) * (u + 1), 4 * m * (m2 + 1), K)


@pytest.mark.parametrize("G,top,T,W,ff", [(8, 2, 20, 256, 320), (32, 4, 24, 512, 128), (4, 2, 16, 64, 192)])
def test_expert_feed_forward(ops, G, top, T, W, ff):
    """the joint call has the bits of its two products (the inner rows are rounded by the second one)"""
    g = torch.Generator(device="cuda").manual_seed(W + ff)
    x = torch.randn(T, W, device="cuda", generator=g)
    ids = torch.rand(T, G, device="cuda", generator=g).topk(top, 1).indices.int()
    off, tok, place = ops.moe_sort(ids, G)
    gate, up = ((torch.randn(G, ff, W, device="cuda", generator=g) * W ** -0.5).bfloat16() for _ in range(2))
    down = (torch.randn(G, W, ff, device="cuda", generator=g) * ff ** -0.5).bfloat16()
    P = T * top
    assert _C.lib.mi_gemm_any_streams(P, ff, W, G)
    one = ops.expert_ff(x, tok, gate, up, down, _C.ACT_SILU, off, P, place)
    a = ops.gemm_any_grouped_act(x, tok, gate, up, _C.ACT_SILU, off, P, None, P)
    assert torch.equal(one, ops.gemm_any_grouped(a, None, down, None, off, P, place, P))
    t, k = 3, 1
    e, xr = int(ids[t, k]), x[3].bfloat16().double()
    inner = torch.nn.functional.silu(gate[e].double() @ xr) * (up[e].double() @ xr)
    want = down[e].double() @ inner
    assert (one[t * top + k].double() - want).norm() <= 2 ** -8 * want.norm()   # (one bf16 rounding of each inner value: 2^-9)
