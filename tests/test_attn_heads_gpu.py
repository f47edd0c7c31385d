"""Decode steps of paged_attention_f32 over bf16 caches (a kv head's query heads as the columns of the score tile) against plain fp64
attention: the head sizes that have a form of their own, value rows in 16-, 4- and 2-byte pieces, pages of any size, several workgroups
per row, long and empty contexts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(H, G, D, Dv, bs, lens, window, kept=0, softcap=0.0, log=False, slope=False, extra=0, latent=False, value_heads=None, seed=0):
    from nanovllm import _C, ops

    g = torch.Generator().manual_seed(seed + D * Dv + bs + len(lens))
    n, pages = len(lens), [max(1, -(-m // bs)) for m in lens]
    Gv = value_heads or G
    total = sum(pages) + 1
    order = torch.randperm(total, generator=g).to(torch.int32)
    table = torch.full((n, max(pages)), -1, dtype=torch.int32)
    at = 0
    for i, m in enumerate(pages):
        table[i, :m] = order[at:at + m]
        at += m
    kc = torch.randn(total, G, bs, D, generator=g).bfloat16()
    ldv = D if latent else Dv + extra
    vc = kc if latent else torch.randn(total, Gv, bs, ldv, generator=g).bfloat16()
    q = torch.randn(n, H * D, generator=g)
    sink = torch.randn(H, generator=g)
    p1, p2 = torch.rand(H, generator=g), torch.rand(H, generator=g)
    scale = D ** -0.5
    want = torch.zeros(n, H, Dv, dtype=torch.float64)
    for i, m in enumerate(lens):
        if m == 0:
            continue
        pg = table[i, :-(-m // bs)].long()
        k = kc[pg].double().permute(1, 0, 2, 3).reshape(G, -1, D)[:, :m].repeat_interleave(H // G, 0)
        v = vc[pg].double().permute(1, 0, 2, 3).reshape(Gv if not latent else G, -1, ldv)[:, :m, :Dv]
        v = v.repeat_interleave(H // v.shape[0], 0)
        s = torch.einsum("hd,hjd->hj", q[i].double().view(H, D), k) * scale
        j = torch.arange(m)
        dist = (m - 1 - j).double()
        if log:
            s = s - p1.double()[:, None] * torch.log1p(p2.double()[:, None] * dist)
        elif slope:
            s = s - p1.double()[:, None] * dist
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        s = s.masked_fill(~((dist < window) | (j < kept)), float("-inf"))
        s = torch.cat([s, sink.double()[:, None]], 1)
        want[i] = torch.einsum("hj,hjd->hd", torch.softmax(s, 1)[:, :-1], v)
    cu = torch.arange(n + 1, dtype=torch.int32).cuda()
    kcd = kc.cuda()
    kind = _C.BIAS_LOG if log else _C.BIAS_SLOPE if slope else _C.BIAS_NONE
    got = ops.paged_attention_f32(q.cuda(), kcd, kcd if latent else vc.cuda(), ldv, table.cuda(), cu,
                                  torch.tensor(lens, dtype=torch.int32).cuda(), H, G, D, Dv, bs, window, scale, kind,
                                  p1.cuda() if log or slope else None, p2.cuda() if log else None, sink=sink.cuda(), softcap=softcap,
                                  value_heads=value_heads, kept=kept)
    live = [i for i, m in enumerate(lens) if m]
    # q and the weights are carried as bf16 hi + lo pairs (16 bits: 2^-17 of each), the sums in fp32
    assert (got.cpu().double().view(n, H, Dv)[live] - want[live]).abs().max() <= 1e-4 * max(1.0, float(want.abs().max()))


RAGGED = [1, 31, 32, 33, 64, 255, 256, 257, 511, 700, 1025, 2049]


@pytest.mark.parametrize("bs", [16, 24, 64])
@pytest.mark.parametrize("H,G,D,Dv", [(16, 8, 128, 128), (8, 1, 256, 256), (4, 2, 64, 128), (20, 1, 128, 128), (4, 2, 256, 128), (6, 3, 96, 64),
                                      (4, 4, 32, 48), (2, 1, 192, 160), (2, 2, 128, 16)])
def test_head_sizes_and_pages(H, G, D, Dv, bs):
    _case(H, G, D, Dv, bs, RAGGED, 1 << 30)
    _case(H, G, D, Dv, bs, RAGGED, 300, seed=1)


@pytest.mark.parametrize("D,Dv", [(128, 128), (256, 256)])
@pytest.mark.parametrize("opts", [dict(kept=5), dict(kept=40), dict(slope=True), dict(log=True), dict(softcap=20.0), dict(softcap=20.0, log=True, kept=3),
                                  dict(extra=8), dict(extra=2), dict(extra=128)])
def test_options(D, Dv, opts):
    _case(8, 2, D, Dv, 32, RAGGED, 200, **opts)


def test_latent_rows_shared_value_heads_and_empty_rows():
    _case(8, 1, 256, 256, 64, RAGGED, 1 << 30, latent=True)
    _case(8, 1, 256, 128, 64, RAGGED, 1 << 30, latent=True)
    _case(8, 4, 128, 128, 16, RAGGED, 1 << 30, value_heads=2)
    _case(8, 4, 128, 128, 16, [0, 77, 0, 1, 300], 1 << 30)


@pytest.mark.parametrize("rows", [1, 2, 7, 16, 17, 33, 70])
def test_rows_that_share_a_launch(rows):
    """one workgroup per (row, kv head) or several, with and without a merge"""
    lens = [1 + (i * 397) % 1500 for i in range(rows)]
    _case(4, 2, 128, 128, 16, lens, 1 << 30)
    _case(8, 1, 256, 256, 16, lens, 1 << 30)
