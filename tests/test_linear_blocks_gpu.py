"""Linear attention with a decayed state over prompt portions, sixteen rows at a time (csrc/delta_blocks.hip), against the recurrence in 64 bits
and against the row-by-row kernel: edges of a block, ragged and empty sequences, states carried from one form to the other, padded key
channels, value columns that fill neither a wave nor a block of the state's layout, decays near 0 and at 1.

Tolerance: an output is a chain of fp32 dot products over D key channels and the rows of its block: each rounds by at most (D + 16) * 2^-24 of
the sum of its terms' magnitudes, taken as 4 times the largest output."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(kind, rows, H, D, Dv):
    from nanovllm import _C

    t = dict(proj=torch.randn(rows, 2 * H * D + H * Dv + 5), f_bias=torch.randn(H * D), lower=torch.rand(H * D) * 0.9, decay=torch.rand(H))
    t["lower"][::3] = 0.0
    t["decay"][0] = 1.0
    if kind == "forget":
        t["proj"][:, 1 + H * D:1 + 2 * H * D] *= 4      # gates from nearly 0 to 1
        acts, code = (_C.ACT_SILU, _C.ACT_NONE, _C.ACT_NONE), _C.DECAY_FORGET
    else:
        acts, code = ((_C.ACT_SILU,) * 3 if kind == "head" else (_C.ACT_NONE,) * 3), _C.DECAY_HEAD
    return t, acts, code


def _call(t, acts, code, H, D, Dv, rows, state, cu, kv, slots, max_rows):
    from nanovllm import _C, ops

    head = code == _C.DECAY_HEAD
    return ops.linear_attention(t["proj"][rows], 1, 1 + H * D, 3 + 2 * H * D, acts, code, t["decay"] if head else None,
                                None if head else t["f_bias"], None if head else t["lower"], None, None, H, state, cu, kv, slots, H, D, Dv,
                                1e-6, max_rows=max_rows)


def _want(t, kind, lens, H, D, Dv):
    p = t["proj"].double()
    silu = torch.nn.functional.silu
    q, k, v = p[:, 1:1 + H * D], p[:, 1 + H * D:1 + 2 * H * D], p[:, 3 + 2 * H * D:3 + 2 * H * D + H * Dv]
    if kind == "forget":
        lo = t["lower"].double()
        g = (lo + (1 - lo) * torch.sigmoid(k + t["f_bias"].double())).view(-1, H, D)
        q, k, v = silu(q).view(-1, H, D), 1 - g, v.view(-1, H, Dv)
    else:
        g = t["decay"].double().view(1, H, 1).expand(p.shape[0], H, D)
        q, k, v = ((silu(x) if kind == "head" else x).view(p.shape[0], H, -1) for x in (q, k, v))
    out, states, r = [], [], 0
    for n in lens:
        S = torch.zeros(H, D, Dv, dtype=torch.float64)
        for i in range(r, r + n):
            S = S * g[i].unsqueeze(-1) + k[i].unsqueeze(-1) * v[i].unsqueeze(-2)
            out.append(torch.einsum("hdv,hd->hv", S, q[i]).reshape(-1))
        r += n
    return torch.stack(out)


def _steps(call, lens, state, chunk, forms):
    n = len(lens)
    starts = [sum(lens[:i]) for i in range(n)]
    done, out, step = [0] * n, None, 0
    while any(d < l for d, l in zip(done, lens)):
        take = [min(l - d, chunk or l) for d, l in zip(done, lens)]
        rows = torch.cat([torch.arange(s + d, s + d + t) for s, d, t in zip(starts, done, take)]).cuda()
        cu = torch.tensor([0] + list(torch.tensor(take).cumsum(0)), dtype=torch.int32).cuda()
        done = [d + t for d, t in zip(done, take)]
        o = call(rows, state, cu, torch.tensor(done, dtype=torch.int32).cuda(), torch.arange(n - 1, -1, -1, dtype=torch.int32).cuda(),
                 forms[step % len(forms)])
        step += 1
        out = torch.zeros(sum(lens), o.shape[1], device="cuda") if out is None else out
        out[rows] = o
    return out


@pytest.mark.parametrize("kind", ["head", "plain", "forget"])
@pytest.mark.parametrize("lens", [(33, 0, 1, 16, 15, 17), (100,), (64, 5)])
@pytest.mark.parametrize("H,D,Dv", [(4, 128, 128), (2, 40, 24), (3, 64, 40), (2, 200, 72), (1, 256, 33)])
def test_linear_attention_by_blocks(kind, lens, H, D, Dv):
    from nanovllm import ops

    torch.manual_seed(sum(lens) + D)
    t, acts, code = _inputs(kind, sum(lens), H, D, Dv)
    want = _want(t, kind, lens, H, D, Dv)
    g = {n: x.cuda() for n, x in t.items()}
    call = lambda *a: _call(g, acts, code, H, D, Dv, *a)
    new = lambda: torch.full((len(lens), ops.linear_attention_state_elems(H, D, Dv)), 7.0, device="cuda")
    s_blocks, s_rows = new(), new()
    got, by_row, mixed = _steps(call, lens, s_blocks, None, [4096]), _steps(call, lens, s_rows, None, [1]), _steps(call, lens, new(), 19, [4096, 1])
    tol = 4 * (D + 16) * 2.0 ** -24 * float(want.abs().max())
    for x in (got, mixed):
        assert (x.cpu().double() - want).abs().max() <= tol
    live = [len(lens) - 1 - i for i, n in enumerate(lens) if n]
    assert (s_blocks[live] - s_rows[live]).abs().max() <= 4 * (D + 16) * 2.0 ** -24 * s_rows[live].abs().max()
    assert all((s_blocks[len(lens) - 1 - i] == 7.0).all() for i, n in enumerate(lens) if n == 0)


@pytest.mark.parametrize("kind", ["head", "forget"])
def test_no_further_from_64_bits_than_row_by_row(kind):
    """rms of the error over a long sequence"""
    from nanovllm import ops

    torch.manual_seed(9)
    H, D, Dv, n = 4, 128, 128, 700
    t, acts, code = _inputs(kind, n, H, D, Dv)
    want = _want(t, kind, [n], H, D, Dv)
    g = {m: x.cuda() for m, x in t.items()}
    err = []
    for form in (4096, 1):
        state = torch.zeros(1, ops.linear_attention_state_elems(H, D, Dv), device="cuda")
        x = _steps(lambda *a: _call(g, acts, code, H, D, Dv, *a), [n], state, None, [form])
        err.append(float((x.cpu().double() - want).pow(2).mean().sqrt()))
    print("rms", kind, err)
    assert err[0] <= err[1]


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("kind", ["head", "forget"])
@pytest.mark.parametrize("at", [0, 5, 21, 32, 66])
def test_values_that_are_not_finite_stay_behind_their_row(kind, where, value, at):
    """the rows in front of it, of its own block too, are what they are without it, and what is not finite behind it is what the row-by-row
    kernel has not finite"""
    from nanovllm import ops

    torch.manual_seed(at)
    n, H, D, Dv = 70, 4, 64, 40
    t, acts, code = _inputs(kind, n, H, D, Dv)
    g = {m: x.cuda() for m, x in t.items()}

    def call(form):
        state = torch.full((2, ops.linear_attention_state_elems(H, D, Dv)), 7.0, device="cuda")
        i32 = lambda *a: torch.tensor(a, dtype=torch.int32).cuda()
        return _call(g, acts, code, H, D, Dv, torch.arange(n).cuda(), state, i32(0, n - 3, n), i32(n - 3, 3), i32(1, 0), form), state

    clean, _ = call(4096)
    assert torch.isfinite(clean).all()
    g["proj"][at, {"q": 1 + 3, "k": 1 + H * D + D + 2, "v": 3 + 2 * H * D + 2 * Dv + 33}[where]] = value
    (got, state), (by_row, row_state) = call(4096), call(1)
    assert torch.equal(got[:at], clean[:at])
    assert torch.equal(torch.isfinite(got), torch.isfinite(by_row))
    assert torch.equal(torch.isfinite(state), torch.isfinite(row_state))
    fine = torch.isfinite(by_row)
    assert (got[fine] - by_row[fine]).abs().max() <= 8 * (D + 16) * 2.0 ** -24 * clean.abs().max()
