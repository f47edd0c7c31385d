"""The row-wise fp32 kernels that read 16 bytes a lane where pointers, strides and widths allow it, and one float at a time otherwise
(csrc/seqmix.hip: layernorm, gated norm-and-add, the experts' sum, the causal convolution): both forms over the same numbers, against
the operation in 64 bits.  Widths: below and at the 256 from which the norms go in pieces, what a thread keeps (4096 by pieces, 1024 by floats) and beyond.

Tolerance: sums of `width` fp32 terms in chains of at most width / 256 + 14 additions, each rounded to 2^-24 of the partial sum; the
results are of order one, so (width / 256 + 32) * 2^-24 * 8 covers sum, root, quotient and the products behind them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from nanovllm import ops as o
    return o


def _off(t):
    """The same rows 4 bytes past a 16-byte border, rows an odd number of floats apart: read one float at a time."""
    base = torch.empty(t.shape[0], t.shape[1] + 3, device="cuda")[:, 1:1 + t.shape[1]] if t.dim() == 2 else \
        torch.empty(t.numel() + 1, device="cuda")[1:]
    return base.copy_(t)


WIDTHS = [4, 36, 252, 256, 260, 1024, 1028, 2048, 4096, 4100, 9000]
ROWS = 5


def _tol(width):
    return (width / 256 + 32) * 2.0 ** -24 * 8


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("add", [False, True])
def test_layernorm_in_pieces(ops, width, add):
    torch.manual_seed(width)
    y, w, b, res = torch.randn(ROWS, width) * 3 + 1, 1 + 0.1 * torch.randn(width), torch.randn(width), torch.randn(ROWS, width)
    want = torch.nn.functional.layer_norm(y.double(), (width,), w.double(), b.double(), 1e-5) + (res.double() if add else 0)
    for place in (lambda t: t.cuda(), lambda t: _off(t.cuda())):
        got = ops.layernorm_f32(place(y), w.cuda(), b.cuda(), 1e-5, add_to=place(res) if add else None)
        assert (got.cpu().double() - want).abs().max() <= _tol(width) * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("nxt", [False, True])
def test_gated_norm_add_in_pieces(ops, width, gate, nxt):
    torch.manual_seed(width + 1)
    res, y, g = (torch.randn(ROWS, width) for _ in range(3))
    w, w2 = 1 + 0.1 * torch.randn(width), 1 + 0.1 * torch.randn(width)
    v = y.double() * (g.double().sigmoid() if gate else 1)
    rms = lambda x: x / (x.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()
    want = res.double() + rms(v) * w.double()
    for place in (lambda t: t.cuda(), lambda t: _off(t.cuda())):
        r = place(res)
        h = ops.gated_norm_add_f32(r, place(y), place(g) if gate else None, w.cuda(), 1e-5, w2.cuda() if nxt else None)
        assert (r.cpu().double() - want).abs().max() <= _tol(width) * want.abs().max()
        if nxt:
            assert (h.cpu().double() - rms(want) * w2.double()).abs().max() <= 2 * _tol(width) * want.abs().max()
        else:
            assert h is None


@pytest.mark.parametrize("width", [4, 36, 1024, 1028, 2060])
@pytest.mark.parametrize("top_k", [1, 3, 4, 5, 8, 9])
def test_sums_of_experts_in_pieces(ops, width, top_k):
    """Both forms add in the same order: equal bits; an identity expert takes the token's own row, untouched parts may hold NaN."""
    torch.manual_seed(width + top_k)
    T, E = 7, 12
    ids = torch.stack([torch.randperm(E + 2)[:top_k] for _ in range(T)]).to(torch.int32)
    wts, h = torch.rand(T, top_k), torch.randn(T, width)
    y = torch.randn(T, top_k, width)
    own = ids >= E
    want = (torch.where(own.unsqueeze(-1), h.unsqueeze(1), y).double() * wts.double().unsqueeze(-1)).sum(1)
    y[own] = float("nan")
    y = y.view(T * top_k, width).cuda()
    got = ops.moe_combine_f32(y, h.cuda(), ids.cuda(), wts.cuda(), E)
    odd = ops.moe_combine_f32(y, _off(h.cuda()), ids.cuda(), wts.cuda(), E)
    assert torch.equal(got, odd)
    assert (got.cpu().double() - want).abs().max() <= top_k * 2.0 ** -24 * 8 * max(1.0, want.abs().max().item())
    if not own.any():
        sh, sg = torch.randn(T, width), torch.randn(T, 1)
        want = want + sg.double().sigmoid() * sh.double()
        got = ops.moe_combine_shared(y, ids.cuda(), wts.cuda(), width, sh.cuda(), sg.cuda())
        odd = ops.moe_combine_shared(y, ids.cuda(), wts.cuda(), width, _off(sh.cuda()), sg.cuda())
        assert torch.equal(got, odd)
        assert (got.cpu().double() - want).abs().max() <= top_k * 2.0 ** -24 * 8 * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("C", [4, 1028])
@pytest.mark.parametrize("lens", [[9], [8, 8], [1, 0, 2, 30, 1, 1, 7], [1] * 70 + [11]])
def test_convolution_of_eight_rows_at_a_time(ops, taps, C, lens):
    """Steps as small as these go a row per workgroup (an odd row distance: always)."""
    assert sum(lens) * C * (32 + len(lens)) < 32 * 800000
    _convolution(ops, taps, C, lens)


@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("C,lens", [(1028, [803]), (1028, [8] * 99 + [9]), (1028, [1, 0, 2, 30, 1, 1, 7] * 20), (1028, [1] * 700 + [11]),
                                    (4, [1] * 2000 + [5] * 400), (4100, [64, 63, 65, 9])])
def test_convolution_of_eight_rows_in_large_steps(ops, taps, C, lens):
    """Eight rows per thread across the sequences' borders against one row per workgroup (an odd row distance): equal bits."""
    assert sum(lens) * C * (32 + len(lens)) >= 32 * 800000
    _convolution(ops, taps, C, lens)


def _convolution(ops, taps, C, lens):
    torch.manual_seed(taps + C + len(lens))
    n, rows = len(lens), sum(lens)
    x, w = torch.randn(rows, C, device="cuda"), torch.randn(C, taps, device="cuda")
    state = torch.randn(n, taps - 1, C, device="cuda")
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32).cuda()
    kv = torch.tensor([l + (i % 2) * 20 for i, l in enumerate(lens)], dtype=torch.int32).cuda()
    slots = torch.arange(n - 1, -1, -1, dtype=torch.int32).cuda()
    for silu in (False, True):
        got = ops.causal_conv(x, w, state, cu, kv, slots, silu=silu, add_input=not silu)
        assert torch.equal(got, ops.causal_conv(_off(x), w, state, cu, kv, slots, silu=silu, add_input=not silu))
        if not silu:
            for i, l in list(enumerate(lens))[-80:]:
                own = x[cu[i]:cu[i + 1]].double()
                past = state[n - 1 - i].double() if i % 2 else torch.zeros_like(state[0]).double()
                full = torch.cat([past, own])
                want = own + sum(w[:, j].double() * full[j:j + l] for j in range(taps))
                assert l == 0 or (got[cu[i]:cu[i + 1]].double() - want).abs().max() <= (taps + 1) * 2.0 ** -24 * 8 * want.abs().max()


@pytest.mark.parametrize("H,G,D,Dv", [(8, 4, 128, 128), (3, 1, 12, 8), (40, 2, 128, 64), (2, 2, 20, 36)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mix", [False, True])
def test_keys_and_values_to_the_pages_in_pieces(ops, H, G, D, Dv, cache, mix):
    """q and k normed over the whole projection, values mixed, rows to the pages (one row without a slot): 16-byte pieces and, from rows
    an odd distance apart, one float at a time (5120 query channels: beyond what a thread keeps)."""
    torch.manual_seed(H * D + Dv)
    T, bs, nq, nk, nv = 7, 4, H * D, G * D, G * Dv
    proj, qw, kw, vf = torch.randn(T, nq + nk + nv), 1 + 0.1 * torch.randn(nq), 1 + 0.1 * torch.randn(nk), torch.randn(T, nv)
    slots = torch.tensor([5, 0, -1, 11, 2, 7, 8], dtype=torch.int32)
    lam = torch.tensor([0.3])
    rms = lambda x, w: x / (x.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w
    q, k, v = proj.double().split([nq, nk, nv], 1)
    v = 0.7 * v + 0.3 * vf.double() if mix else v
    q, k = rms(q, qw.double()), rms(k, kw.double())
    for place in (lambda t: t.cuda(), lambda t: _off(t.cuda())):
        p = place(proj)
        kc, vc = (torch.full((3, G, bs, d), 9.0, dtype=cache, device="cuda") for d in (D, Dv))
        ops.swa_prepare(p, 0, nq, nq + nk, qw.cuda(), kw.cuda(), 1e-5, place(vf) if mix else None, lam.cuda() if mix else None, kc, vc,
                        slots.cuda(), H, G, D, Dv, bs)
        tol = _tol(max(nq, nk)) * 4
        assert (p[:, :nq].cpu().double() - q).abs().max() <= tol
        assert (p[:, nq + nk:].cpu().double() - v).abs().max() <= tol
        used = torch.zeros(3 * bs, dtype=torch.bool)
        for t, s in enumerate(slots.tolist()):
            if s >= 0:
                used[s] = True
                for c, ref, d in ((kc, k, D), (vc, v, Dv)):
                    got, want = c[s // bs, :, s % bs].cpu().double(), ref[t].view(G, d)
                    assert ((got - want).abs() <= tol + (2.0 ** -8 * want.abs() if cache == torch.bfloat16 else 0)).all()
        for c in (kc, vc):
            assert (c.permute(0, 2, 1, 3).reshape(3 * bs, -1).cpu()[~used] == 9.0).all()


@pytest.mark.parametrize("rows,H,Dv", [(4096, 4, 128), (5461, 3, 100), (16385, 1, 64), (8192, 2, 20)])
@pytest.mark.parametrize("gate", [False, True])
def test_head_norms_four_at_a_time(ops, rows, H, Dv, gate):
    """From 16384 (row, head) pairs on four per wave (5461 x 3: one short of it), in place."""
    from nanovllm import _C
    torch.manual_seed(rows)
    o, z, w = torch.randn(rows, H * Dv + 5), torch.randn(rows, H * Dv), 1 + 0.1 * torch.randn(Dv)
    v = o[:, :H * Dv].double().view(rows, H, Dv)
    want = (v / (v.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()).reshape(rows, -1) * (z.double().sigmoid() if gate else 1)
    got = o.cuda()
    ops.head_norm_gate(got[:, :H * Dv], z.cuda() if gate else None, _C.ACT_SIGMOID, w.cuda(), H, Dv, 1e-5)
    assert (got[:, :H * Dv].cpu().double() - want).abs().max() <= _tol(Dv) * want.abs().max()
    assert torch.equal(got[:, H * Dv:].cpu(), o[:, H * Dv:])
