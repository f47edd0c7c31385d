"""Decode attention with the sequences' workgroups in order of their contexts (context_order, paged_attn_decode_fused(order=...)): the order
itself, and results and cache rows the same bits as without it, for every group size, ragged, equal and empty contexts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 64, 65, 200, 1000, 1024])
def test_order(n):
    from nanovllm import ops

    g = torch.Generator().manual_seed(n)
    lens = torch.randint(0, 40 if n % 2 else 3000, (n,), generator=g, dtype=torch.int32)
    got = ops.context_order(lens.cuda(), 8).cpu()
    want = sorted(range(n), key=lambda i: (-int(lens[i]), i))
    assert got[:, 0].tolist() == want and torch.equal(got[:, 1], lens[got[:, 0].long()])
    assert ops.context_order(lens[:32].cuda(), 8) is None and ops.context_order(torch.zeros(1025, dtype=torch.int32).cuda(), 8) is None


@pytest.mark.parametrize("H,G", [(16, 8), (8, 8), (32, 8), (64, 8), (16, 1)])
@pytest.mark.parametrize("norm", [True, False])
def test_attention_in_order(H, G, norm):
    from nanovllm import ops

    n, bs = (40, 16) if G == 8 else (300, 32)
    g = torch.Generator(device="cuda").manual_seed(H)
    lens = [1 + (i * 367) % 1100 for i in range(n)]
    lens[3] = lens[17] = 0          # rows of a captured step's padding
    lens[5] = lens[6] = lens[7]
    lens[9], lens[10], lens[11] = 16, 17, 128
    pages = [-(-m // bs) for m in lens]
    total = sum(pages) + 1
    order = torch.randperm(total, generator=torch.Generator().manual_seed(1)).int()
    table, at = torch.full((n, max(pages)), -1, dtype=torch.int32), 0
    for i, m in enumerate(pages):
        table[i, :m] = order[at:at + m]
        at += m
    kc, vc = (torch.randn(total, G, bs // 16, 16 * 128, device="cuda", generator=g).bfloat16() for _ in range(2))
    qkv = torch.randn(n, (H + 2 * G) * 128, device="cuda", generator=g).bfloat16()
    qw, kw = (torch.randn(128, device="cuda", generator=g).mul(0.1).add(1).bfloat16() if norm else None for _ in range(2))
    pos = torch.tensor([max(m - 1, 0) for m in lens], device="cuda")
    cos_sin = torch.randn(1200, 128, device="cuda", generator=g)
    slots = torch.tensor([[int(table[i, (m - 1) // bs]), (m - 1) % bs] if m else [-1, -1] for i, m in enumerate(lens)], dtype=torch.int32).cuda()
    ctx = torch.tensor(lens, dtype=torch.int32).cuda()

    def run(o):
        k, v = kc.clone(), vc.clone()
        y = ops.paged_attn_decode_fused(qkv, qw, kw, 1e-6, pos, cos_sin, slots, k, v, table.cuda(), ctx, H, G, bs, 128 ** -0.5, order=o)
        return y, k, v

    o = ops.context_order(ctx, G)
    assert o is not None
    (a, ka, va), (b, kb, vb) = run(None), run(o)
    assert torch.equal(ka, kb) and torch.equal(va, vb)
    assert torch.equal(a, b)
    assert not bool(b[3].any()) and not bool(b[17].any())
