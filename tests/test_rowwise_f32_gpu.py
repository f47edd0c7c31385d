"""The row-wise fp32 kernels that read 16 bytes a lane where pointers, strides and widths allow it, and one float at a time otherwise
(csrc/seqmix.hip: layernorm, gated norm-and-add, the experts' sum, the causal convolution): both forms over the same numbers, against
the operation in 64 bits.  Widths: one piece, less than a workgroup's, what a thread keeps (4096 by pieces, 1024 by floats) and beyond.

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


WIDTHS = [4, 36, 1024, 1028, 2048, 4096, 4100, 9000]
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
    """Eight rows per thread across the sequences' borders against one row per workgroup (an odd row distance): equal bits."""
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
            for i, l in enumerate(lens):
                own = x[cu[i]:cu[i + 1]].double()
                past = state[n - 1 - i].double() if i % 2 else torch.zeros_like(state[0]).double()
                full = torch.cat([past, own])
                want = own + sum(w[:, j].double() * full[j:j + l] for j in range(taps))
                assert l == 0 or (got[cu[i]:cu[i + 1]].double() - want).abs().max() <= (taps + 1) * 2.0 ** -24 * 8 * want.abs().max()
