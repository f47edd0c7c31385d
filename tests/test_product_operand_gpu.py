"""A norm's second output, its rows rounded to bf16, and the products that read it in place of rounding the rows themselves: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from nanovllm import ops
    return ops


def _same(a, b):
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


# one piece per thread and several, the last one part-filled, more than a thread keeps, widths and strides that are no whole pieces
@pytest.mark.parametrize("width,pad", [(64, 0), (256, 0), (1024, 0), (1028, 4), (1027, 0), (1024, 1), (2048, 8), (4160, 0), (5121, 0)])
def test_norms_write_both(ops, width, pad):
    g = torch.Generator().manual_seed(width + pad)
    rows = 37
    wide = lambda: torch.randn(rows, width + pad, generator=g).to(DEV)[:, :width]
    vec = lambda: torch.randn(width, generator=g).to(DEV)
    y, res, gate, w, b, nxt = wide(), wide(), wide(), vec(), vec(), vec()
    guard = torch.full((rows + 1, width), 7.0, dtype=torch.bfloat16, device=DEV)
    xb = guard[:rows]
    for add in (False, True):
        want = ops.layernorm_f32(y, w, b, 1e-6, add_to=res.clone() if add else None)
        got = ops.layernorm_f32(y, w, b, 1e-6, add_to=res.clone() if add else None, rounded=xb)
        assert _same(got.contiguous(), want.contiguous()) and torch.equal(xb, want.bfloat16())
    for gp in (gate, None):
        r1, r2 = res.clone(), res.clone()
        want = ops.gated_norm_add_f32(r1, y, gp, w, 1e-6, nxt)
        got = ops.gated_norm_add_f32(r2, y, gp, w, 1e-6, nxt, xb)
        assert _same(r1, r2) and _same(got, want) and torch.equal(xb, want.bfloat16())
    assert bool((guard[rows] == 7.0).all())


@pytest.mark.parametrize("rows,N,K", [(512, 1024, 1024), (513, 200, 192), (777, 4100, 1024), (2049, 2048, 2048), (9, 1024, 1024), (600, 30, 64), (600, 1023, 128)])
def test_products_read_rounded_rows(ops, rows, N, K):
    g = torch.Generator().manual_seed(rows + N)
    x, w, b = torch.randn(rows, K, generator=g).to(DEV), torch.randn(N, K, generator=g).bfloat16().to(DEV), torch.randn(N, generator=g).to(DEV)
    xb = x.bfloat16()
    assert _same(ops.gemm_any(x, w, rounded=xb), ops.gemm_any(x, w))
    assert _same(ops.gemm_any_act(x, w, bias=b, rounded=xb), ops.gemm_any_act(x, w, bias=b))
    f32 = w.float()
    assert _same(ops.gemm_any(x, f32, rounded=xb), ops.gemm_any(x, f32))   # fp32 weights: the rows as they are


@pytest.mark.parametrize("tokens,E,top,ff,W", [(600, 16, 2, 128, 256), (700, 32, 4, 512, 1024), (512, 8, 1, 192, 128)])
def test_experts_read_rounded_rows(ops, tokens, E, top, ff, W):
    from nanovllm import _C

    g = torch.Generator().manual_seed(tokens)
    ids = torch.rand(tokens, E, generator=g).topk(top, 1).indices.to(torch.int32).to(DEV)
    offsets, pair_token, pair_index = ops.moe_sort(ids, E)
    x = torch.randn(tokens, W, generator=g).to(DEV)
    gate, up = (torch.randn(E, ff, W, generator=g).bfloat16().to(DEV) for _ in range(2))
    down = torch.randn(E, W, ff, generator=g).bfloat16().to(DEV)
    args = (pair_token, gate, up, down, _C.ACT_SILU, offsets, tokens * top, pair_index)
    assert _same(ops.expert_ff(x, *args, rounded=x.bfloat16()), ops.expert_ff(x, *args))
