"""The channel-wise delta rule of prompt portions, sixteen rows at a time (csrc/delta_blocks.hip), against the recurrence in 64 bits and
against the row-by-row kernel: edges of a block (15, 16, 17, 33 rows), ragged and empty sequences, states carried from one form to
the other, key channels that are padded (40, 200), value columns that fill neither a wave (24) nor a block of the state's layout (40),
decays near 0 and at 1.

Tolerance: every output is a chain of fp32 dot products over D key channels and the block's rows: each rounds by at most (D + 16) * 2^-24
of the sum of its terms' magnitudes, taken as 4 times the largest read-out before its norm (unit keys; states are sums of such terms)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from nanovllm import ops as o
    return o


def _steps(call, lens, state, chunk, forms):
    """The sequences' rows through the op: all at once (chunk None) or `chunk` rows of every sequence at a time; forms: the most rows
    of a sequence as the op is told in the steps' turn (a large number: blocks, 1: row by row)."""
    n = len(lens)
    starts = [sum(lens[:i]) for i in range(n)]
    done, out, step = [0] * n, None, 0
    while any(d < l for d, l in zip(done, lens)):
        take = [min(l - d, chunk or l) for d, l in zip(done, lens)]
        rows = torch.cat([torch.arange(s + d, s + d + t) for s, d, t in zip(starts, done, take)]).cuda()
        cu = torch.tensor([0] + list(torch.tensor(take).cumsum(0)), dtype=torch.int32).cuda()
        done = [d + t for d, t in zip(done, take)]
        o = call(rows, state, cu, torch.tensor(done, dtype=torch.int32).cuda(),
                 torch.arange(n - 1, -1, -1, dtype=torch.int32).cuda(), forms[step % len(forms)])
        step += 1
        out = torch.zeros(sum(lens), o.shape[1], device="cuda") if out is None else out
        out[rows] = o
    return out


def _check(got, rowwise, want, scale, D, what):
    tol = 4 * (D + 16) * 2.0 ** -24
    e, e_row = (((x.double() - want).abs() / scale).max().item() for x in (got, rowwise))
    assert torch.isfinite(got).all() and e <= tol, (what, e, e_row, tol)


LENS = [(33, 0, 1, 16, 15, 17), (100,), (64, 5)]


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (2, 2, 40, 24), (3, 1, 64, 40), (2, 1, 200, 72)])
def test_channel_delta_by_blocks(ops, lens, H, G, D, Dv):
    torch.manual_seed(sum(lens) + D)
    rows, eps = sum(lens), 1e-6
    width = 2 * G * D + H * Dv + 8
    qkv = torch.randn(rows, width)
    beta, gate = torch.randn(rows, H), torch.randn(rows, H * Dv)
    decay = torch.randn(rows, H * D) * 3           # decays from nearly 0 to 1
    dt, a_log, w = torch.randn(H * D), torch.randn(H) * 0.5, 1 + 0.1 * torch.randn(Dv)
    g = {k: v.cuda() for k, v in dict(qkv=qkv, beta=beta, gate=gate, decay=decay, dt=dt, a_log=a_log, w=w).items()}

    def call(r, state, cu, kv, slots, max_rows):
        return ops.channel_delta(g["qkv"][r], 0, G * D, 2 * G * D, g["beta"][r], g["decay"][r], g["dt"], g["a_log"], g["gate"][r], g["w"],
                                 state, cu, kv, slots, H, G, D, Dv, eps, max_rows)

    want, r = torch.zeros(rows, H, Dv, dtype=torch.float64), 0
    q, k, v = (qkv.double()[:, o:o + n] for o, n in ((0, G * D), (G * D, G * D), (2 * G * D, H * Dv)))
    unit = lambda x: x.view(rows, G, D) / (x.view(rows, G, D).pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()
    q, k = (unit(x).repeat_interleave(H // G, 1) for x in (q, k))
    f = torch.exp(-a_log.double().exp()[:, None] * torch.nn.functional.softplus(decay.double() + dt.double()).view(rows, H, D))
    for n in lens:
        S = torch.zeros(H, D, Dv, dtype=torch.float64)
        for t in range(r, r + n):
            S = S * f[t].unsqueeze(-1)
            u = beta.double()[t].sigmoid()[:, None] * (v[t].view(H, Dv) - (S * k[t].unsqueeze(-1)).sum(1))
            S = S + k[t].unsqueeze(-1) * u.unsqueeze(1)
            want[t] = (S * q[t].unsqueeze(-1)).sum(1) * D ** -0.5
        r += n
    rms = (want.pow(2).mean(-1, keepdim=True) + eps).sqrt()
    scale = (want.abs().max() / rms).expand(-1, -1, Dv).reshape(rows, -1)   # (the read-out norm divides a head by its own size)
    want = (want / rms * w.double()).view(rows, -1) * gate.double().sigmoid()
    new = lambda: torch.full((len(lens), ops.channel_delta_state_elems(H, D, Dv)), 7.0, device="cuda")
    s_blocks, s_rows = new(), new()
    got = _steps(call, lens, s_blocks, None, [4096])
    by_row = _steps(call, lens, s_rows, None, [1])
    mixed = _steps(call, lens, new(), 19, [4096, 1])
    for name, x in (("blocks", got), ("blocks and rows", mixed)):
        _check(x.cpu(), by_row.cpu(), want, scale, D, f"delta {lens} {(H, G, D, Dv)} {name}")
    live = [len(lens) - 1 - i for i, n in enumerate(lens) if n]   # (slots are handed out in reverse; an empty sequence's stays as it was)
    assert (s_blocks[live] - s_rows[live]).abs().max() <= 4 * (D + 16) * 2.0 ** -24 * s_rows[live].abs().max()
    assert all((s_blocks[len(lens) - 1 - i] == 7.0).all() for i, n in enumerate(lens) if n == 0)


@pytest.mark.parametrize("lens", [tuple(i * 37 % 23 for i in range(70)), (40,) * 65, (0,) * 64 + (33, 0, 34), (1,) * 3 + (90,),
                                  tuple(i % 3 for i in range(511)) + (35,), tuple(i % 3 for i in range(512)) + (35,)])
@pytest.mark.parametrize("H,G,D,Dv", [(3, 1, 64, 40), (2, 2, 128, 96), (4, 2, 200, 72)])
def test_sequences_in_the_order_of_their_rows(ops, lens, H, G, D, Dv):
    """every sequence walked once: more than a wave looks at, as many as are put in order and one more, equal ones, empty ones; 256 channels
    with 32 columns a workgroup and (more of them than CUs) 64, which are beyond the state's columns here"""
    test_channel_delta_by_blocks(ops, lens, H, G, D, Dv)



@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "decay", "beta"])
@pytest.mark.parametrize("at", [0, 5, 21, 32, 66])
def test_values_that_are_not_finite_stay_behind_their_row(ops, where, value, at):
    """A NaN or an infinity in a row: the rows in front of it, of its own block too, are what they are without it, and what is not finite
    behind it is what the row-by-row kernel has not finite."""
    torch.manual_seed(at)
    n, H, G, D, Dv, eps = 70, 4, 2, 64, 40, 1e-6
    t = dict(qkv=torch.randn(n, 2 * G * D + H * Dv), beta=torch.randn(n, H), gate=torch.randn(n, H * Dv), decay=torch.randn(n, H * D),
             dt=torch.randn(H * D), a_log=torch.randn(H) * 0.5, w=1 + 0.1 * torch.randn(Dv))
    g = {k: v.cuda() for k, v in t.items()}

    def call(max_rows):
        state = torch.full((2, ops.channel_delta_state_elems(H, D, Dv)), 7.0, device="cuda")
        o = ops.channel_delta(g["qkv"], 0, G * D, 2 * G * D, g["beta"], g["decay"], g["dt"], g["a_log"], g["gate"], g["w"], state,
                              torch.tensor([0, n - 3, n], dtype=torch.int32).cuda(), torch.tensor([n - 3, 3], dtype=torch.int32).cuda(),
                              torch.tensor([1, 0], dtype=torch.int32).cuda(), H, G, D, Dv, eps, max_rows)
        return o, state

    clean, clean_state = call(4096)
    assert torch.isfinite(clean).all()
    name, col = {"q": ("qkv", 3), "k": ("qkv", G * D + D + 2), "v": ("qkv", 2 * G * D + 2 * Dv + 33), "decay": ("decay", D + 9), "beta": ("beta", 1)}[where]
    g[name][at, col] = -value if where == "decay" else value   # (an infinite decay of 0 is a plain number)
    (got, state), (by_row, row_state) = call(4096), call(1)
    assert torch.equal(got[:at], clean[:at])
    assert torch.equal(torch.isfinite(got), torch.isfinite(by_row))
    assert torch.equal(torch.isfinite(state), torch.isfinite(row_state))
    fine = torch.isfinite(by_row)
    assert (got[fine] - by_row[fine]).abs().max() <= 8 * (D + 16) * 2.0 ** -24 * clean.abs().max() * (clean.abs().max() / clean.pow(2).mean().sqrt())
    assert torch.equal(got[n - 3:][torch.isfinite(got[n - 3:])], clean[n - 3:][torch.isfinite(got[n - 3:])])
