"""The experts' first product with its rows gathered by the tile kernels' feed: the bits of the product over rows that a pass wrote out in
the experts' order, at every tile size and with ragged, empty and one-row experts."""
import pytest
import torch

from nanovllm import _C, ops

pytestmark = pytest.mark.gpu


def _written_out(h, tok, gate, up, down, act, off, pairs, place, limit, scale, scale_rows):
    """mi_expert_ff: the rows of x are not named, so the operand pass gathers"""
    G, ff, W = gate.shape
    n = _C.lib.mi_expert_ff_bytes(pairs, G, ff, W, 1, int(act))
    assert n
    scratch, y = torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty(pairs, W, device="cuda")
    p = lambda t: 0 if t is None else t.data_ptr()
    rc = _C.lib.mi_expert_ff(p(h), h.stride(0), p(tok), p(gate), p(up), p(down), int(act), float(limit), p(scale), p(scale_rows), p(off),
                             p(place), pairs, G, ff, W, p(scratch), n, p(y), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return y


@pytest.mark.parametrize("E,top,T,W,ff,want", [(8, 2, 500, 256, 128, 128), (32, 4, 300, 512, 320, 64), (24, 6, 3000, 1280, 640, 256),
                                               (5, 1, 700, 128, 192, 128), (64, 8, 160, 256, 256, 64), (3, 3, 257, 64, 256, 128)])
@pytest.mark.parametrize("act,limit", [(_C.ACT_SILU, 0.0), (_C.ACT_GELU_TANH, 0.0), (_C.ACT_CLAMPED_GLU, 7.0)])
def test_gathered_rows(E, top, T, W, ff, want, act, limit):
    g = torch.Generator(device="cuda").manual_seed(T + ff)
    h = torch.randn(T, W + 4, device="cuda", generator=g)[:, :W]
    lean = torch.rand(T, E, device="cuda", generator=g) + torch.linspace(0, 0.8, E, device="cuda")   # (ragged experts)
    lean[:, 0] = -1   # nobody's
    lean[:, 1] = -1
    lean[0, 1] = 9    # one row
    ids = lean.topk(top, 1).indices.int()
    wts = torch.rand(T, top, device="cuda", generator=g)
    off, tok, place = ops.moe_sort(ids, E)
    gate, up = (torch.randn(E, ff, W, device="cuda", generator=g).mul(W ** -0.5).bfloat16() for _ in range(2))
    down = torch.randn(E, W, ff, device="cuda", generator=g).mul(ff ** -0.5).bfloat16()
    scale = wts if act == _C.ACT_CLAMPED_GLU else None
    rows = place if scale is not None else None
    P = T * top
    first = _C.lib.mi_gemm_any_tile_rows(P, ff, W, E, 1, int(act))
    second = _C.lib.mi_gemm_any_tile_rows(P, W, ff, E, 0, _C.ACT_NONE)
    assert min(first, second) == want and not _C.lib.mi_gemm_any_streams(P, ff, W, E)
    a = ops.expert_ff(h, tok, gate, up, down, act, off, P, place, limit, scale, rows)
    assert torch.equal(a, _written_out(h, tok, gate, up, down, act, off, P, place, limit, scale, rows))
    b = ops.expert_ff(torch.cat([h, h[:1]]), tok, gate, up, down, act, off, P, place, limit, scale, rows)   # (top 1: more rows than pairs)
    assert torch.equal(a, b)
