"""Projections of a few rows with the launch in front of them in their operand load (csrc/gemm_few.hip): the bits of the two launches
they stand for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(*shape, std=1.0, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, device="cuda", generator=g) * std).to(dtype)


def _pack(w, fp8):
    from nanovllm import ops

    return ops.pack_weight_fp8(w) if fp8 else ops.pack_weight(w)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("K,nsplit", [(512, 2), (768, 4), (1024, 4), (1024, 8)])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
def test_norm_few(rows, K, nsplit, fp8):
    from nanovllm import ops

    parts = _rand(nsplit, rows, K, dtype=torch.float32, seed=rows)
    res, norm_w = _rand(rows, K, seed=7), _rand(K, std=0.1, seed=8) + 1
    for n, silu in ((16, False), (1024, False), (96, True)):
        w = _pack(_rand(n, K, std=0.05, seed=n), fp8)
        assert ops.norm_few_takes(rows, nsplit, w, silu)
        got, got_res = ops.gemm_norm_few(parts, res, norm_w, 1e-6, w, silu)
        x, want_res = ops.add_rmsnorm_splitk(parts, res, norm_w, 1e-6)
        assert torch.equal(got_res, want_res) and torch.equal(got, ops.gemm_packed(x, w, silu_mul=silu)), (n, silu)


def test_norm_few_refuses():
    from nanovllm import ops

    w = _pack(_rand(64, 1024), False)
    assert not ops.norm_few_takes(ops.FEW_ROWS_MAX + 1, 4, w, False) and not ops.norm_few_takes(1, 3, w, False)
    with pytest.raises(Exception):
        ops.gemm_norm_few(_rand(4, 5, 1024, dtype=torch.float32), _rand(5, 1024), _rand(1024), 1e-6, w)


@pytest.mark.parametrize("fp8", [False, True])
# 8, 8, 4, 12, 16 and 8 waves; the last with four splits at four rows
@pytest.mark.parametrize("heads,kv_heads,ksplit", [(16, 8, 4), (8, 2, 2), (8, 8, 4), (12, 3, 2), (16, 8, 2), (16, 16, 4)])
@pytest.mark.parametrize("lens", [[1], [16], [33, 0], [300, 17, 1], [128, 2047, 64, 1], [5, 700, 31, 32]])
def test_merge_few(lens, heads, kv_heads, ksplit, fp8):
    """Contexts of no, one and many splits with keys; a length of 0 (a padding row of a captured batch) gives a zero row"""
    from nanovllm import ops

    B, D, block = len(lens), 128, 16
    pages = [max(1, -(-n // block)) for n in lens]
    total = sum(pages)
    kc, vc = (_rand(*ops.kv_cache_shape(total, kv_heads, block), seed=s) for s in (1, 2))
    table = torch.full((B, max(pages)), 0, dtype=torch.int32)
    order, at, slots = torch.randperm(total, generator=torch.Generator().manual_seed(3)).int(), 0, []
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
        last = lens[i] - 1
        slots.append([int(table[i, last // block]), last % block] if lens[i] else [-1, 0])
    table, slots = table.cuda(), torch.tensor(slots, dtype=torch.int32, device="cuda")
    ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
    pos = (ctx.long() - 1).clamp(min=0)
    qkv = _rand(B, (heads + 2 * kv_heads) * D, seed=4)
    qw, kw = _rand(D, std=0.1, seed=5) + 1, _rand(D, std=0.1, seed=6) + 1
    ang = torch.arange(4096).float().view(-1, 1) / 1e4 ** (torch.arange(64).float() / 64)
    cs = torch.cat([ang.cos(), ang.sin()], 1).contiguous().cuda()
    w = _pack(_rand(256, heads * D, std=0.03, seed=9), fp8)
    args = (qw, kw, 1e-6, pos, cs, slots)
    rest = (table, ctx, heads, kv_heads, block, D ** -0.5)
    k2, v2 = kc.clone(), vc.clone()
    want = ops.gemm_packed_splitk(ops.paged_attn_decode_fused(qkv, *args, k2, v2, *rest), w, ksplit)
    assert ops.merge_few_takes(B, kv_heads, w, ksplit)
    got = ops.paged_attn_few_proj(qkv, *args, kc, vc, *rest, w, ksplit)
    assert torch.equal(kc, k2) and torch.equal(vc, v2) and torch.equal(got, want)


def test_merge_few_refuses():
    from nanovllm import ops

    w = _pack(_rand(256, 2048), False)
    assert not ops.merge_few_takes(1, 8, w, 1)     # 32 waves
    assert not ops.merge_few_takes(1, 8, w, 16)    # 2 waves
    assert not ops.merge_few_takes(ops.FEW_ROWS_MAX + 1, 8, w, 4)
    assert not ops.merge_few_takes(4, 64, w, 4)    # contexts in one piece
