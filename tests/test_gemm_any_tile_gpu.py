"""Projections of the 32-bit-residual families on the tile kernels (mi_gemm_any_tile): edges of row, feature and
group tiles, both kernels, every epilogue, scattered rows, against a float64 statement over the rounded operands.

Bound: the operands' products are exact in fp32, the sum over K carries at most K roundings of 2^-24 of the absolute sum, the
epilogue a handful more; activations are 1.13-Lipschitz at most (gelu, silu), relu^2 and the clamped pair scale with their
arguments - so: error <= (K + 16) * 2^-24 * (what the same expression gives on absolute values) + 1e-6."""
import pytest
import torch

from nanovllm import _C, ops

pytestmark = pytest.mark.gpu


def _ref(z, z2, act, limit):
    if act == _C.ACT_CLAMPED_GLU:
        g, u = z.clamp(max=limit), z2.clamp(-limit, limit)
        return g * torch.sigmoid(1.702 * g) * (u + 1)
    a = {_C.ACT_NONE: lambda t: t, _C.ACT_SILU: torch.nn.functional.silu, _C.ACT_GELU_ERF: torch.nn.functional.gelu,
         _C.ACT_GELU_TANH: lambda t: torch.nn.functional.gelu(t, approximate="tanh"), _C.ACT_RELU2: lambda t: t.clamp(min=0) ** 2}[act](z)
    return a if z2 is None else a * z2


def _close(got, want, size, K):
    err = (got.double() - want).abs()
    bound = (K + 16) * 2.0 ** -24 * size + 1e-6
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("M,N,K", [(65, 64, 64), (17, 68, 512), (256, 128, 64), (257, 132, 128), (511, 260, 192), (1030, 644, 320)])
@pytest.mark.parametrize("act,dual", [(_C.ACT_NONE, False), (_C.ACT_GELU_ERF, False), (_C.ACT_RELU2, False), (_C.ACT_SILU, True),
                                      (_C.ACT_GELU_TANH, True)])
def test_plain_rows(tile, M, N, K, act, dual):
    g = torch.Generator(device="cuda").manual_seed(M + N + K + act)
    x = torch.randn(M, K + 3, device="cuda", generator=g)[:, :K]   # rows that do not start on 16 bytes
    w, w2 = (torch.randn(N, K, device="cuda", generator=g).mul(K ** -0.5).bfloat16() for _ in range(2))
    bias, bias2 = torch.randn(N, device="cuda", generator=g), torch.randn(N, device="cuda", generator=g)
    w2, bias2 = (w2, bias2) if dual else (None, None)
    out = torch.full((M + 1, N), 7.0, device="cuda")
    ops._tile_gemm(ops._tile_operand(x, tile), tile, w, w2, out[:M], act, bias=bias, bias2=bias2, alpha=0.5)
    xr = x.bfloat16().double()
    z = xr @ w.double().T + bias
    z2 = xr @ w2.double().T + bias2 if dual else None
    s = xr.abs() @ w.double().abs().T + bias.abs()
    s2 = xr.abs() @ w2.double().abs().T + bias2.abs() if dual else 1.0
    size = 2 * s * (s if act == _C.ACT_RELU2 else 1.0) * s2
    _close(out[:M], 0.5 * _ref(z, z2, act, 0.0), size, K)
    assert bool((out[M] == 7.0).all())


@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("counts", [(300, 0, 1, 128, 129), (0, 0, 256, 257), (64,) * 8, (5, 700), (1, 0, 65, 3, 64, 2)])
@pytest.mark.parametrize("act", [_C.ACT_SILU, _C.ACT_CLAMPED_GLU])
def test_grouped_rows(tile, counts, act):
    G, N, K, T = len(counts), 196, 128, 211
    g = torch.Generator(device="cuda").manual_seed(sum(counts) + act)
    P = sum(counts) + 9   # the last nine rows belong to no group
    x = torch.randn(T, K, device="cuda", generator=g)
    rows = torch.randint(0, T, (P,), device="cuda", generator=g, dtype=torch.int32)
    rows[sum(counts):] = 1 << 30   # (never looked at)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    w, w2 = (torch.randn(G, N, K, device="cuda", generator=g).mul(K ** -0.5).bfloat16() for _ in range(2))
    scale = torch.rand(P, device="cuda", generator=g) if act == _C.ACT_CLAMPED_GLU else None
    y = torch.full((P, N), 7.0, device="cuda")
    operand = ops._tile_operand(x, tile, rows, off, G, P)
    ops._tile_gemm(operand, tile, w, w2, y, act, G, place, limit=1.5, row_scale=scale, row_scale_rows=place if scale is not None else None)
    y16 = torch.zeros((P, N), device="cuda", dtype=torch.bfloat16)
    ops._tile_gemm(operand, tile, w, w2, y16, act, G, place, limit=1.5, row_scale=scale, row_scale_rows=place if scale is not None else None)
    want, size = torch.full((P, N), 7.0, device="cuda", dtype=torch.float64), torch.ones(P, N, device="cuda", dtype=torch.float64)
    for e in range(G):
        r = slice(int(off[e]), int(off[e + 1]))
        xr, at = x[rows[r].long()].bfloat16().double(), place[r].long()
        f = scale[at].double().unsqueeze(1) if scale is not None else 1.0
        z, z2 = xr @ w[e].double().T * f, xr @ w2[e].double().T * f
        want[at] = _ref(z, z2, act, 1.5)
        size[at] = 4 * (xr.abs() @ w[e].double().abs().T) * (xr.abs() @ w2[e].double().abs().T + 1)
    _close(y, want, size, K)
    done = place[:sum(counts)].long()
    assert torch.equal(y16[done], y[done].bfloat16())


@pytest.mark.parametrize("act,limit", [(_C.ACT_SILU, 0.0), (_C.ACT_CLAMPED_GLU, 7.0)])
def test_expert_pair_takes_the_same_bits_as_two_products(act, limit):
    E, top, T, W, ff = 8, 2, 500, 256, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    h = torch.randn(T, W, device="cuda", generator=g)
    ids = torch.randint(0, E, (T, top), device="cuda", generator=g, dtype=torch.int32)
    wts = torch.rand(T, top, device="cuda", generator=g)
    off, tok, place = ops.moe_sort(ids, E)
    gate, up = (torch.randn(E, ff, W, device="cuda", generator=g).mul(W ** -0.5).bfloat16() for _ in range(2))
    down = torch.randn(E, W, ff, device="cuda", generator=g).mul(ff ** -0.5).bfloat16()
    scale = wts if act == _C.ACT_CLAMPED_GLU else None
    a = ops.gemm_any_grouped_glu(h, tok, gate, up, act, limit, scale, place if scale is not None else None, off, T * top, None, T * top)
    two = ops.gemm_any_grouped(a, None, down, None, off, T * top, place, T * top)
    one = ops.expert_ff(h, tok, gate, up, down, act, off, T * top, place, limit, scale, place if scale is not None else None)
    assert ops._tile_rows(T * top, gate, up, act, False, E) and torch.equal(one, two)


@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("counts", [(200,) * 8, (9, 0, 300, 1)])
def test_bound_on_one_groups_rows(counts, gathered):
    """rows_max bounds ONE group; the product covers the rows of all of them"""
    G, N, K, T, P = len(counts), 68, 64, 111, sum(counts)
    g = torch.Generator(device="cuda").manual_seed(P)
    x = torch.randn(T if gathered else P, K, device="cuda", generator=g)
    rows = torch.randint(0, T, (P,), device="cuda", generator=g, dtype=torch.int32) if gathered else None
    xs = (x[rows.long()] if gathered else x).bfloat16().double()
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    w, w2 = (torch.randn(G, N, K, device="cuda", generator=g).mul(K ** -0.5).bfloat16() for _ in range(2))
    z, z2, s, s2 = (torch.empty(P, N, device="cuda", dtype=torch.float64) for _ in range(4))
    for e in range(G):
        r = slice(int(off[e]), int(off[e + 1]))
        at = place[r].long()
        z[at], z2[at] = xs[r] @ w[e].double().T, xs[r] @ w2[e].double().T
        s[at], s2[at] = xs[r].abs() @ w[e].double().abs().T, xs[r].abs() @ w2[e].double().abs().T
    most = max(counts)
    _close(ops.gemm_any_grouped(x, rows, w, None, off, most, place, P), z, s, K)
    _close(ops.gemm_any_grouped_act(x, rows, w, None, _C.ACT_RELU2, off, most, place, P), z.clamp(min=0) ** 2, 2 * s * s, K)
    _close(ops.gemm_any_grouped_glu(x, rows, w, w2, _C.ACT_CLAMPED_GLU, 1.5, None, None, off, most, place, P),
           _ref(z, z2, _C.ACT_CLAMPED_GLU, 1.5), 4 * s * (s2 + 1), K)


# what the dispatch picks for large work: the persistent kernel over several tiles per workgroup (more than 2 x 256 of them: the next
# tile's group is fetched under the running one's products), 128-row tiles on the two-stage ring (more than 256 of them), 64-row tiles
# of 128 features for one weight (more than 1024 of 64)
LARGE = [(256, 24, 1028, 64, False, 33000), (256, 24, 516, 128, True, 33000), (256, 0, 1284, 64, False, 30000), (256, 0, 644, 64, True, 26000),
         (128, 12, 516, 64, False, 9000), (128, 12, 260, 64, True, 9000), (128, 0, 516, 128, False, 9000), (64, 64, 2052, 64, False, 1500),
         (64, 64, 1028, 256, True, 1500), (64, 0, 2052, 64, False, 3000)]


@pytest.mark.parametrize("tile,G,N,K,dual,rows", LARGE)
def test_more_tiles_than_the_chip_holds(tile, G, N, K, dual, rows):
    g = torch.Generator(device="cuda").manual_seed(N + rows)
    act = _C.ACT_SILU if dual else _C.ACT_NONE
    row_tiles = rows // tile + G if G else -(-rows // tile)
    wide = {256: 128 if dual else 256, 128: 64 if dual else 128, 64: 64}[tile]
    assert row_tiles * -(-N // wide) > {256: 512, 128: 256, 64: 1024}[tile]
    x = torch.randn(rows, K, device="cuda", generator=g)
    place = torch.randperm(rows, device="cuda", generator=g).to(torch.int32)
    if G:   # ragged, every fifth group empty, the last rows in none
        share = torch.rand(G, generator=torch.Generator().manual_seed(G)) + 0.1
        share[::5] = 0
        counts = (share / share.sum() * (rows - 100)).long().tolist()
        off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device="cuda")
    else:
        counts, off = [rows], None
    w, w2 = (torch.randn(max(G, 1), N, K, device="cuda", generator=g).mul(K ** -0.5).bfloat16() for _ in range(2))
    y = torch.full((rows, N), 7.0, device="cuda")
    ww, ww2 = (w, w2) if G else (w[0], w2[0])
    ops._tile_gemm(ops._tile_operand(x, tile, None, off, G, rows), tile, ww, ww2 if dual else None, y, act, G, place)
    lo = 0
    for e, n in enumerate(counts):
        xr, at = x[lo:lo + n].bfloat16().double(), place[lo:lo + n].long()
        z, s = xr @ w[e].double().T, xr.abs() @ w[e].double().abs().T
        if dual:
            z2, s2 = xr @ w2[e].double().T, xr.abs() @ w2[e].double().abs().T
            z, s = torch.nn.functional.silu(z) * z2, 4 * s * (s2 + 1)
        _close(y[at], z, s, K)
        lo += n
    assert bool((y[place[lo:].long()] == 7.0).all())


@pytest.mark.parametrize("rows,N,K,G,dual,want", [(65536, 768, 2048, 64, True, 256), (65536, 2048, 768, 64, False, 256), (1024, 2048, 768, 64, False, 64),
                                                  (256, 2048, 768, 64, False, 64), (8192, 2048, 2048, 0, False, 256), (2048, 768, 2048, 32, True, 128),
                                                  (1536, 512, 4096, 32, True, 128), (1536, 512, 4096, 32, False, 64), (1280, 512, 2048, 20, True, 64),
                                                  (31580, 384, 256, 16, False, 128), (4660, 1664, 3456, 32, True, 256), (17664, 320, 192, 64, True, 128)])
def test_rule_reaches_the_large_forms(rows, N, K, G, dual, want):
    assert _C.lib.mi_gemm_any_tile_rows(rows, N, K, G, int(dual), _C.ACT_SILU if dual else _C.ACT_NONE) == want


@pytest.mark.parametrize("rows,N,K", [(130, 256, 64), (255, 512, 128), (257, 768, 64), (700, 256, 320)])
@pytest.mark.parametrize("form", ["plain", "bias", "groups", "pair"])
def test_whole_feature_tiles_of_the_persistent_kernel(form, rows, N, K):
    """The 256-row kernel's short epilogue (whole feature tiles, nothing on rows or results; two weights: bf16 results): the same bits as
    the 128-row kernel's, row for row, scattered and bounded by the groups; nothing written beside them."""
    g = torch.Generator(device="cuda").manual_seed(rows + N + K)
    G = 3 if form in ("groups", "pair") else 0
    x = torch.randn(rows, K, device="cuda", generator=g)
    w, w2 = (torch.randn(max(G, 1), N, K, device="cuda", generator=g).mul(K ** -0.5).bfloat16() for _ in range(2))
    w, w2 = (w, w2) if G else (w[0], w2[0])
    bias = torch.randn(N, device="cuda", generator=g) if form == "bias" else None
    cut = rows // 3
    off = torch.tensor([0, cut, cut, rows - rows // 7], dtype=torch.int32, device="cuda") if G else None
    place = torch.randperm(rows, device="cuda", generator=g).to(torch.int32) if G else None
    outs = []
    for tile in (256, 128):
        out = torch.full((rows + 1, N), 7.0, device="cuda", dtype=torch.bfloat16 if form == "pair" else torch.float32)
        operand = ops._tile_operand(x, tile, None, off, G, rows) if G else ops._tile_operand(x, tile)
        ops._tile_gemm(operand, tile, w, w2 if form == "pair" else None, out[:rows], _C.ACT_SILU if form == "pair" else _C.ACT_NONE, G,
                       place, bias=bias)
        outs.append(out)
    assert torch.equal(*outs)
    done = rows - rows // 7 if G else rows
    assert int((outs[0] != 7.0).any(1).sum()) == done and bool((outs[0][rows] == 7.0).all())
    if form in ("plain", "bias"):
        xr, b = x.bfloat16().double(), 0.0 if bias is None else bias
        size = xr.abs() @ w.double().abs().T + (0.0 if bias is None else bias.abs())
        _close(outs[0][:rows], xr @ w.double().T + b, size, K)


@pytest.mark.parametrize("tile", [64, 256])
def test_silu_of_large_arguments(tile):
    """0 and z to an ulp where the exponential is out of range, finite everywhere; to an ulp also where the quotient's reciprocal is no normal
    number (-88.5 .. -87.5); below that the exponential overflows, as expf's did"""
    z = torch.tensor([0.0, -0.0, 80.0, -80.0, 87.0, 88.0, -87.0, -87.5, -88.0, -88.5, 104.5, -104.5, 1e30, -1e30, 3e38, -3e38], device="cuda").bfloat16().float().repeat(5)
    x, w, w2 = torch.zeros(z.numel(), 64, device="cuda"), torch.zeros(128, 64, device="cuda"), torch.zeros(128, 64, device="cuda")
    x[:, 0], x[:, 1], w[:, 0], w2[:, 1] = z, 1.0, 1.0, 1.0
    out = torch.empty(z.numel(), 128, device="cuda")
    ops._tile_gemm(ops._tile_operand(x, tile), tile, w.bfloat16(), w2.bfloat16(), out, _C.ACT_SILU)
    want = torch.nn.functional.silu(z.double()).unsqueeze(1)
    low = torch.where((z < -88.72) & (z > -120), 3e-37, 0.0).unsqueeze(1)   # (z / inf)
    assert bool(((out.double() - want).abs() <= 4 * 2.0 ** -24 * want.abs() + low).all())
