"""What the order of a decode step's contexts is made for, and what takes it.  The library is not called."""
import pytest
import torch

from nanovllm import _C, ops


class _Recorder:
    def __init__(self, lib):
        self.lib, self.calls = lib, []

    def __getattr__(self, name):
        if name not in ("mi_context_order", "mi_paged_attn_decode_fused_ordered"):
            return getattr(self.lib, name)
        return lambda *a: self.calls.append((name, a)) or 0


@pytest.fixture
def calls(monkeypatch):
    rec = _Recorder(_C.lib)
    monkeypatch.setattr(ops, "lib", rec)
    monkeypatch.setattr(ops, "require_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "stream", lambda: 0)
    return rec.calls


def test_shallow_models_make_no_order(calls):
    lens = torch.full((64,), 500, dtype=torch.int32)
    assert ops.context_order(lens, 8, 1) is None and ops.context_order(lens, 8, ops.CONTEXT_ORDER_LAYERS - 1) is None and not calls
    assert ops.context_order(lens, 8, ops.CONTEXT_ORDER_LAYERS) is not None and ops.context_order(lens, 8) is not None and len(calls) == 2
    assert ops.context_order(lens, 4, 28) is None and len(calls) == 2


def test_an_order_that_is_not_on_the_gpu_is_refused(monkeypatch, calls):
    """its pointer goes to the kernel as the others do"""
    asked = []
    monkeypatch.setattr(ops, "require_gpu", lambda *a: asked.extend(a))
    n, H, G, bs = 40, 16, 8, 16
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32)
    order, cache = i32(n, 2), torch.zeros(*ops.kv_cache_shape(1, G, bs), dtype=torch.bfloat16)
    ops.paged_attn_decode_fused(torch.zeros(n, (H + 2 * G) * 128, dtype=torch.bfloat16), None, None, 1e-6, torch.zeros(n, dtype=torch.int64), torch.zeros(4, 128),
                                i32(n, 2), cache, cache, i32(n, 1), i32(n), H, G, bs, 1.0, out=torch.zeros(n, H * 128, dtype=torch.bfloat16),
                                workspace=torch.zeros(16, dtype=torch.uint8), order=order)
    assert any(t is order for t in asked) and calls[-1][1][-2] == order.data_ptr()
