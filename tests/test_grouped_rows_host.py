"""Grouped products take `rows_max` as a bound on ONE group's rows: the operand buffer and the tile table of the tile path have to be
sized for the rows of all groups.  The library calls are recorded, not made."""
import pytest
import torch

from nanovllm import _C, ops


class _Recorder:
    """mi_gemm_any_operand / mi_gemm_any_tile / mi_expert_ff_tokens recorded, everything else the library's own"""

    def __init__(self, lib):
        self.lib, self.calls = lib, {}

    def __getattr__(self, name):
        if name not in ("mi_gemm_any_operand", "mi_gemm_any_tile", "mi_expert_ff_tokens"):
            return getattr(self.lib, name)
        return lambda *a: self.calls.__setitem__(name, a) or 0


@pytest.fixture
def recorded(monkeypatch):
    rec = _Recorder(_C.lib)
    monkeypatch.setattr(ops, "lib", rec)
    monkeypatch.setattr(ops, "require_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "stream", lambda: 0)
    return rec.calls


@pytest.mark.parametrize("name", ["gemm_any_grouped", "gemm_any_grouped_act", "gemm_any_grouped_glu"])
@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("counts", [(200,) * 8, (9, 0, 300, 1)])
def test_rows_of_all_groups(monkeypatch, recorded, name, gathered, counts):
    G, N, K, total = len(counts), 64, 64, sum(counts)
    made = []
    empty = torch.empty
    monkeypatch.setattr(ops.torch, "empty", lambda *a, **k: made.append(empty(*a, **k)) or made[-1])
    w = torch.zeros(G, N, K, dtype=torch.bfloat16)
    off = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32)
    x = torch.zeros(17 if gathered else total, K)
    x_rows = torch.zeros(total, dtype=torch.int32) if gathered else None
    y_rows = torch.arange(total, dtype=torch.int32)
    most = max(counts)
    if name == "gemm_any_grouped":
        ops.gemm_any_grouped(x, x_rows, w, None, off, most, y_rows, total)
    elif name == "gemm_any_grouped_act":
        ops.gemm_any_grouped_act(x, x_rows, w, None, _C.ACT_NONE, off, most, y_rows, total)
    else:
        ops.gemm_any_grouped_glu(x, x_rows, w, None, _C.ACT_NONE, 0.0, None, None, off, most, y_rows, total)
    operand, tile = recorded["mi_gemm_any_operand"], recorded["mi_gemm_any_tile"]
    tile_rows, rows = operand[5], operand[6]
    assert rows >= total and tile[16] >= total
    xb = next(t for t in made if t.data_ptr() == operand[8])
    table = next(t for t in made if t.data_ptr() == operand[9])
    assert xb.shape[0] >= total
    assert table.numel() >= 4 + 4 * sum(-(-c // tile_rows) for c in counts)


def test_few_rows_per_group_stay_on_the_kernel_that_does_not_round_them():
    w = torch.zeros(64, 64, 64, dtype=torch.bfloat16)
    assert ops._grouped_tile_rows(512, 9, w, None, _C.ACT_NONE, False)
    assert not ops._grouped_tile_rows(512, 8, w, None, _C.ACT_NONE, False)


def test_soft_capped_products_have_no_256_row_tiles():
    """mi_gemm_any_tile: tiles of 256 rows are the persistent kernel's, which has no soft-capped form (no rows: nothing is launched)"""
    p, run = 1 << 20, _C.lib.mi_gemm_any_tile
    args = lambda act, tile, rows: (p, None, tile, p, None, None, None, act, 0.0, None, None, 0, p, 0, 8192, None, rows, 8192, 64, 30.0, None)
    assert run(*args(_C.ACT_SOFTCAP, 256, 0)) == -2
    for act, tile in ((_C.ACT_SOFTCAP, 128), (_C.ACT_SOFTCAP, 64), (_C.ACT_NONE, 256)):
        assert run(*args(act, tile, 0)) == 0


def test_expert_feed_forward_takes_the_operands_that_the_two_products_take(recorded):
    """a scale per pair is read as it lies in memory: strided ones are refused by both routes"""
    G, T, top, W, ff = 4, 50, 2, 256, 256
    x, gate, down = torch.zeros(T, W), torch.zeros(G, ff, W, dtype=torch.bfloat16), torch.zeros(G, W, ff, dtype=torch.bfloat16)
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32)
    args = (x, i32(T * top), gate, gate, down, _C.ACT_CLAMPED_GLU, i32(G + 1), T * top, i32(T * top), 7.0)
    ops.expert_ff(*args, torch.ones(T, top), i32(T * top))
    assert "mi_expert_ff_tokens" in recorded
    recorded.clear()
    with pytest.raises(AssertionError):
        ops.expert_ff(*args, torch.ones(T, 2 * top)[:, :top], i32(T * top))
    assert not recorded


def test_few_pairs_of_small_experts_stay_on_the_general_kernels(recorded):
    """both products or neither: the line is the same whichever of the two a product is"""
    rows = lambda P, N, K, G, dual=False: _C.lib.mi_gemm_any_tile_rows(P, N, K, G, int(dual), _C.ACT_SILU if dual else _C.ACT_RELU2)
    for P, ff, width, G in ((16, 256, 256, 8), (96, 256, 512, 16), (32, 256, 512, 32), (24, 192, 512, 128), (32, 512, 1024, 8)):
        assert not rows(P, ff, width, G, True) and not rows(P, width, ff, G) and not _C.lib.mi_expert_ff_bytes(P, G, ff, width, 1, _C.ACT_SILU)
    for P, ff, width, G in ((65, 256, 256, 8), (48, 256, 512, 32), (128, 256, 512, 16), (16, 512, 1024, 32), (16, 768, 2048, 64), (96, 512, 1024, 8)):
        assert rows(P, ff, width, G, True) and rows(P, width, ff, G) and _C.lib.mi_expert_ff_bytes(P, G, ff, width, 1, _C.ACT_SILU)
