"""The sum of the experts' outputs where they are more than the caches hold (fetched past them): the plain weighted sum, identity experts among
the picks, one to eight parts, a row and a column that do not fill a workgroup."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,top,W", [(8300, 8, 1028), (16500, 4, 1032), (33000, 2, 1024), (65600, 1, 1028), (8190, 8, 1024), (9000, 7, 1100)])
def test_combine(T, top, W):
    from nanovllm import ops

    g = torch.Generator(device="cuda").manual_seed(T)
    E = 12
    y = torch.randn(T * top, W, device="cuda", generator=g)
    h = torch.randn(T, W, device="cuda", generator=g)
    ids = torch.randint(0, E + 2, (T, top), device="cuda", generator=g, dtype=torch.int32)   # E and E + 1: the row itself
    wts = torch.rand(T, top, device="cuda", generator=g)
    got = ops.moe_combine_f32(y, h, ids, wts, E)
    want = torch.zeros(T, W, device="cuda")
    for k in range(top):   # the parts in order, a fused multiply-add each
        part = torch.where((ids[:, k] >= E).unsqueeze(1), h, y.view(T, top, W)[:, k])
        want = torch.addcmul(want, part, wts[:, k:k + 1])
    # |parts| below 6 and weights below 1: a step rounds a sum below 6 * top by 2^-24 of it on either side, top steps
    assert (got - want).abs().max() <= 2.0 ** -23 * 6 * top * top
