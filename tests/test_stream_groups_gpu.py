"""Streamed products of experts whose shares are uneven (csrc/gemm_any.hip: gemm_any_stream_groups_kernel): the rows beyond a group's first sixteen go to
workgroups of their own - more groups than a wave has lanes, pieces that the workgroups take behind one another, all rows in one group - against
float64 over the rounded operands (bound: tests/test_gemm_any_stream_gpu.py), and the time that uneven shares take."""
import pytest
import torch

from nanovllm import _C

pytestmark = pytest.mark.gpu


def _off(counts):
    return torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("counts,bound", [((300,) + (0,) * 39, None), ((0,) * 30 + (16, 17, 32, 33, 0, 1, 15, 200), None), ((5, 97) * 35, None), ((100,) * 12, 100),
                                          ((40, 0, 31, 64, 9), 64), ((9,) * 3, None)])
@pytest.mark.parametrize("K,N", [(64, 36), (192, 4100)])
def test_uneven_groups(counts, bound, K, N):
    from nanovllm import ops

    G, P, T = len(counts), sum(counts), 29
    g = torch.Generator(device="cuda").manual_seed(P + N)
    x = torch.randn(T, K, device="cuda", generator=g)
    w, w2 = ((torch.randn(G, N, K, device="cuda", generator=g) * K ** -0.5).bfloat16() for _ in range(2))
    rows = torch.randint(0, T, (P,), device="cuda", generator=g, dtype=torch.int32)
    place = torch.randperm(P, device="cuda", generator=g).to(torch.int32)
    off = _off(counts)
    y = [torch.empty(P, N, device="cuda") for _ in range(2)]
    for out, second in zip(y, (None, w2)):   # (the C entry: the wrapper's rule looks at the average share)
        rc = _C.lib.mi_gemm_any_grouped_act(x.data_ptr(), K, rows.data_ptr(), w.data_ptr(), None if second is None else second.data_ptr(), _C.DTYPE_BF16,
                                            _C.ACT_NONE if second is None else _C.ACT_SILU, off.data_ptr(), G, bound or min(P, 8 * G), out.data_ptr(), N,
                                            place.data_ptr(), N, K, 0, ops.stream())
        assert rc == 0
    for e, n in enumerate(counts):
        r = slice(int(off[e]), int(off[e]) + n)
        xr, at = x[rows[r].long()].bfloat16().double(), place[r].long()
        z, m = xr @ w[e].double().T, xr.abs() @ w[e].double().abs().T
        z2, m2 = xr @ w2[e].double().T, xr.abs() @ w2[e].double().abs().T
        room = (K + 16) * 2.0 ** -24
        assert bool(((y[0][at].double() - z).abs() <= room * m + 1e-6).all()), e
        assert bool(((y[1][at].double() - torch.nn.functional.silu(z) * z2).abs() <= room * 3 * m * (m2 + 1) + 1e-6).all()), e


def test_a_step_on_one_expert_takes_no_longer_than_one_on_all():
    """757 pairs of 128 experts of 512 x 512, on one of them or shared evenly: the latter reads 128 times the weights (as one workgroup's walk per
    expert the former took five times as long)"""
    from nanovllm import ops

    E, P, W = 128, 757, 512
    x = torch.randn(P, W, device="cuda")
    gate, up, down = (torch.randn(E, W, W, device="cuda").mul(0.04).bfloat16() for _ in range(3))
    times = []
    for ids in (torch.zeros(P, 1), torch.arange(P).view(P, 1) % E):
        off, tok, place = ops.moe_sort(ids.int().cuda(), E)
        best = float("inf")
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(20):
                ops.expert_ff(x, tok, gate, up, down, _C.ACT_SILU, off, P, place)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
    assert times[0] <= 2 * times[1], times
