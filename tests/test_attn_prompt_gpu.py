"""Attention of prompt portions (csrc/attn_prompt.hip): the forms its images, tiles and page look-ups branch on, against float64.

Bounds.  bf16 pages: q and the weights enter the products as hi + lo pairs (2^-17 of each), the rest is fp32; fp32 pages: fp32
throughout, scores in units of ln 2 (2^-23 of a score's size in a weight's exponent).  With |scores| <= 30: 2e-5 of the largest value
on bf16 pages, 1e-5 on fp32 pages."""
import math

import pytest
import torch

from nanovllm import _C, ops

pytestmark = pytest.mark.gpu


def _case(dtype, H, G, D, Dv, block, seqs, window=2 ** 31 - 1, kept=0, chunk=0, softcap=0.0, sink=False, bias=_C.BIAS_NONE, vik=False,
          gate=False, value_heads=None, pad=0):
    g = torch.Generator(device="cuda").manual_seed(H * 131 + D * 7 + Dv + block + len(seqs))
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    Gv = value_heads or G
    pages = [-(-(a + n) // block) for a, n in seqs]
    order = torch.randperm(sum(pages) + 1, device="cuda", generator=g).int()
    table = torch.full((len(seqs), max(pages)), -1, dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    k_cache = torch.full((len(order), G, block, D), float("nan"), device="cuda").to(dtype)   # rows nobody wrote stay NaN
    v_cache = k_cache if vik else torch.full((len(order), Gv, block, Dv + pad), float("nan"), device="cuda").to(dtype)
    ks, vs = [], []
    for i, (a, n) in enumerate(seqs):
        p = torch.arange(a + n, device="cuda")
        k = rnd(a + n, G, D).to(dtype)
        k_cache[table[i, p // block].long(), :, p % block] = k
        if not vik:
            v = rnd(a + n, Gv, Dv).to(dtype)
            v_cache[table[i, p // block].long(), :, p % block, :Dv] = v
        ks.append(k.double())
        vs.append(k.double()[..., :Dv] if vik else v.double())
    rows = sum(n for _, n in seqs)
    q, gt = rnd(rows, H * D), rnd(rows, H * Dv) if gate else None
    cu = torch.tensor([0] + list(torch.tensor([n for _, n in seqs]).cumsum(0)), dtype=torch.int32, device="cuda")
    kv = torch.tensor([a + n for a, n in seqs], dtype=torch.int32, device="cuda")
    sk = rnd(H) if sink else None
    p1, p2 = (torch.rand(H, device="cuda", generator=g), torch.rand(H, device="cuda", generator=g)) if bias == _C.BIAS_LOG else (None, None)
    scale = D ** -0.5
    got = ops.paged_attention_f32(q, k_cache, v_cache, D if vik else Dv + pad, table, cu, kv, H, G, D, Dv, block, window, scale, bias, p1, p2,
                                  gate=gt, sink=sk, softcap=softcap, chunk=chunk, kept=kept, value_heads=Gv)
    want = torch.empty(rows, H, Dv, dtype=torch.float64, device="cuda")
    for i, (a, n) in enumerate(seqs):
        qq = q[int(cu[i]):int(cu[i + 1])].double().view(n, H, D)
        pos, key = torch.arange(a, a + n, device="cuda").view(-1, 1), torch.arange(a + n, device="cuda").view(1, -1)
        dist = pos - key
        seen = (dist >= 0) & (((dist < window) & ((pos // chunk == key // chunk) if chunk else True)) | (key < kept))
        for h in range(H):
            s = qq[:, h] @ ks[i][:, h // (H // G)].T * scale
            if bias == _C.BIAS_SLOPE:
                s = s - 2.0 ** (-8.0 * (h + 1) / H) * dist
            elif bias == _C.BIAS_LOG:
                s = s - p1[h].double() * torch.log1p(p2[h].double() * dist.clamp(min=0))
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            s = s.masked_fill(~seen, -math.inf)
            if sink:
                s = torch.cat([s, sk[h].double().expand(n, 1)], 1)
            want[int(cu[i]):int(cu[i + 1]), h] = torch.softmax(s, 1)[:, :a + n] @ vs[i][:, h // (H // Gv)]
    want = want.view(rows, H * Dv)
    if gate:
        want = want * torch.sigmoid(gt.double())
    tol = (2e-5 if dtype == torch.bfloat16 else 1e-5) * float(want.abs().max())
    assert float((got.double() - want).abs().max()) <= tol


SEQS = ((0, 1), (130, 70), (0, 33), (17, 1), (31, 2))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv", [(6, 2, 64, 64), (5, 1, 64, 128), (8, 8, 128, 128), (4, 4, 96, 48), (7, 1, 256, 192), (2, 1, 32, 256),
                                      (130, 1, 32, 16)])
def test_head_shapes(dtype, H, G, D, Dv):
    _case(dtype, H, G, D, Dv, 16, SEQS, gate=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("block", [8, 16, 48, 64, 256])
def test_page_sizes(dtype, block):
    _case(dtype, 4, 2, 64, 64, block, SEQS, window=50, bias=_C.BIAS_SLOPE)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("block", [8, 24])
@pytest.mark.parametrize("D,Dv,vik", [(64, 128, False), (128, 112, False), (192, 256, False), (256, 224, True)])
def test_head_sizes_over_pages_of_any_size(dtype, block, D, Dv, vik):
    _case(dtype, 4, 2, D, Dv, block, SEQS, window=50, vik=vik)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("seqs", [((0, 33),), ((0, 64), (0, 40)), ((0, 65), (3, 60)), ((0, 128), (60, 40)), ((0, 129), (0, 40))])
@pytest.mark.parametrize("D,Dv,vik", [(160, 128, False), (128, 192, False), (256, 256, True)])
def test_wide_heads_over_few_keys(dtype, seqs, D, Dv, vik):
    """both sides of the line beyond which fp32 heads of more than 128 channels go to the matrix cores"""
    _case(dtype, 6, 2, D, Dv, 16, seqs, vik=vik, sink=True, gate=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", [dict(window=1), dict(window=40, kept=5), dict(window=64, kept=70), dict(chunk=48), dict(chunk=33, kept=3),
                                  dict(softcap=5.0, sink=True), dict(bias=_C.BIAS_LOG, sink=True), dict(value_heads=1), dict(kept=500)])
def test_masks_and_biases(dtype, form):
    _case(dtype, 4, 2, 64, 128, 32, SEQS + ((200, 97),), **form)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,seqs", [(6, 6, [(i * 37 % 90, (i * 53) % 48) for i in range(100)]), (12, 6, [(40, 700), (0, 0), (3, 257), (0, 1000)] * 3),
                                      (24, 1, [(0, 300)] * 10 + [(500, 61)] * 9), (8, 8, [(i % 3, 64 + i % 2) for i in range(64)]),
                                      (130, 5, [(0, 0)] * 63 + [(7, 129), (0, 127)] * 2 + [(i, 1) for i in range(60)])])
def test_more_tiles_than_the_chip_holds(dtype, H, G, seqs):
    """the longest walks first, over all sequences: every tile once, whatever ends, equal ends, empty sequences and numbers of sequences"""
    _case(dtype, H, G, 32, 32, 16, seqs)


@pytest.mark.parametrize("block", [16, 24])
@pytest.mark.parametrize("D,Dv", [(64, 64), (48, 32)])
@pytest.mark.parametrize("seqs,window", [([(90, 3)] * 40, 2 ** 31 - 1), ([(0, 700), (30, 600)], 64), ([(0, 700), (30, 600)], 2 ** 31 - 1),
                                         ([(i, 40 + 7 * i) for i in range(30)], 2 ** 31 - 1)])
def test_small_fp32_heads_with_one_workgroup_per_cu_and_with_two(block, D, Dv, seqs, window):
    """both sides of the line: a few hundred like walks, a few hundred unlike ones, and many"""
    _case(torch.float32, 14, 7, D, Dv, block, seqs, window=window)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("step", [2.0, 7.9, 8.1, 40.0])
def test_scores_that_grow_along_the_keys(dtype, step):
    """maxima that the reference point follows at once, later or never: keys whose scores rise by `step` powers of two per 32 keys"""
    n, D, block = 160, 32, 16
    k = torch.zeros(10, 1, block, D, device="cuda")
    p = torch.arange(n, device="cuda").view(10, 1, block)
    k[..., 0] = (p // 32) * step            # (integers and tenths: bf16 rounds them as the oracle reads them)
    k, v = k.to(dtype), torch.randn(10, 1, block, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).to(dtype)
    q = torch.zeros(n, D, device="cuda")
    q[:, 0] = torch.linspace(-1, 1, n, device="cuda")
    table = torch.arange(10, device="cuda").int().view(1, 10)
    cu, kv = torch.tensor([0, n], dtype=torch.int32, device="cuda"), torch.tensor([n], dtype=torch.int32, device="cuda")
    got = ops.paged_attention_f32(q, k, v, D, table, cu, kv, 1, 1, D, D, block, 2 ** 31 - 1, math.log(2))
    s = (q.double() @ k.double().view(n, D).T * math.log(2)).masked_fill(torch.ones(n, n, device="cuda").triu(1).bool(), -math.inf)
    want = torch.softmax(s, 1) @ v.double().view(n, D)
    # (scores of up to 160: 2^-17 of their size in a weight's exponent on bf16 pages, 2^-22 on fp32 pages, as the module's bounds say)
    tol = (2e-5 if dtype == torch.bfloat16 else 1e-5) * max(1.0, 4 * step / 30) * float(want.abs().max())
    assert float((got.double() - want).abs().max()) <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,Dv", [(256, 256), (224, 160)])
def test_values_inside_the_key_rows(dtype, D, Dv):
    _case(dtype, 16, 1, D, Dv, 64, SEQS, vik=True, sink=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pad", [1, 2, 4, 6, 8])
@pytest.mark.parametrize("H,G,D,Dv,block", [(4, 2, 64, 64, 16), (6, 1, 128, 48, 24), (2, 2, 256, 256, 64)])
def test_value_rows_of_any_stride(dtype, pad, H, G, D, Dv, block):
    """even strides of bf16 value rows stay on the matrix cores, odd ones go element by element"""
    _case(dtype, H, G, D, Dv, block, SEQS, window=60, pad=pad, gate=True)


@pytest.mark.parametrize("pad", [2, 6])
@pytest.mark.parametrize("H,G,D,Dv,block", [(4, 2, 192, 96, 16), (8, 1, 256, 16, 64), (4, 4, 64, 128, 24)])
def test_narrow_value_rows_of_even_strides_over_long_walks(pad, H, G, D, Dv, block):
    """value heads of at most half the image's 256 channels: every request of a step's values counts in the ring's waits"""
    _case(torch.bfloat16, H, G, D, Dv, block, ((1500, 70), (900, 33)), pad=pad)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("H,G,D,Dv,vik,window,kept", [(4, 2, 64, 64, False, 2 ** 31 - 1, 0), (8, 4, 128, 128, False, 50, 3), (3, 1, 256, 256, True, 40, 0),
                                                      (2, 2, 96, 48, False, 64, 0)])
def test_keys_and_values_that_are_not_finite_reach_the_rows_that_see_them(dtype, value, where, H, G, D, Dv, vik, window, kept):
    """one such key or value row at position 40 of 150: rows in front of it, and rows whose window has passed it, are as without it"""
    if vik and where == "v":
        pytest.skip("the values are the keys")
    n, bad, block = 150, 40, 16
    g = torch.Generator(device="cuda").manual_seed(D)
    k, v = (torch.randn(10, G, block, d, device="cuda", generator=g).to(dtype) for d in (D, Dv))
    v = k if vik else v
    q = torch.randn(n, H * D, device="cuda", generator=g)
    table = torch.randperm(10, device="cuda", generator=g).int().view(1, 10)
    cu, kv = torch.tensor([0, n], dtype=torch.int32, device="cuda"), torch.tensor([n], dtype=torch.int32, device="cuda")

    def call():
        return ops.paged_attention_f32(q, k, v, Dv, table, cu, kv, H, G, D, Dv, block, window, D ** -0.5, kept=kept)

    clean = call()
    (k if where == "k" else v)[table[0, bad // block].long(), G - 1, bad % block, 5] = value
    got = call()
    pos = torch.arange(n, device="cuda")
    sees = (pos >= bad) & (pos - bad < window)
    heads = (torch.arange(H, device="cuda") // (H // G) == G - 1).repeat_interleave(Dv)
    channel = torch.arange(H * Dv, device="cuda") % Dv == 5
    hit = sees.view(-1, 1) & (heads & channel if where == "v" else heads).view(1, -1)
    tol = 2 * (2e-5 if dtype == torch.bfloat16 else 1e-5) * float(clean.abs().max())   # (two results, each within the bound above)
    assert torch.isfinite(got[~hit]).all() and float((got - clean)[~hit].abs().max()) <= tol
    if where == "v" or value != value:   # (an infinite key may just weigh nothing: -inf)
        assert not torch.isfinite(got[hit]).any()
