"""Where a decode step of a few rows has its norms and the merge of its contexts' splits in the next projection's operand load."""
import pytest
import torch

from nanovllm import ops


def _w(n, k, fp8=False):
    return ops.Fp8Weight(torch.empty(0), torch.empty(0), (n, k)) if fp8 else torch.empty(n, k, dtype=torch.bfloat16, device="meta")


@pytest.mark.parametrize("nsplit,n,k,silu,fp8,pays", [(4, 4096, 1024, False, False, True), (4, 8192, 1024, False, True, True), (4, 12288, 1024, False, False, False),
                                                      (8, 4096, 1024, False, False, True), (8, 6144, 1024, False, False, False), (4, 6144, 1024, True, False, True),
                                                      (4, 6144, 1024, True, True, False), (4, 12288, 1024, True, False, False), (8, 6144, 1024, True, False, False),
                                                      (8, 8192, 512, False, False, True), (8, 16384, 512, False, False, False), (4, 8192, 768, False, False, True),
                                                      (8, 16384, 512, True, True, True), (4, 4096, 2048, False, False, False)])
def test_norm(nsplit, n, k, silu, fp8, pays):
    for rows in (1, 2, 3, 4):
        assert ops.norm_few_pays(rows, nsplit, _w(n, k, fp8), silu) == pays
    assert not ops.norm_few_pays(ops.FEW_ROWS_MAX + 1, nsplit, _w(n, k, fp8), silu)


@pytest.mark.parametrize("rows,heads,kv_heads,n,ksplit,pays", [(1, 16, 8, 2048, 2, True), (2, 16, 8, 2048, 2, True), (3, 16, 8, 2048, 2, False), (4, 32, 8, 1024, 4, False),
                                                               (4, 16, 8, 1024, 4, True), (3, 12, 4, 768, 2, True), (4, 8, 8, 1024, 4, True), (5, 8, 8, 1024, 4, False)])
def test_merge(rows, heads, kv_heads, n, ksplit, pays):
    assert ops.merge_few_pays(rows, kv_heads, _w(n, heads * 128), ksplit) == pays


def test_prefill_attention_of_few_rows_rule():
    """The rule counts an XCD's workgroups (fewer pairs than XCDs leave the others idle) and, beyond its places, asks whether the walks
    differ.  Steps measured on both sides of the line."""
    from nanovllm import _C

    takes = lambda seqs, hq, hkv, q, keys: bool(_C.lib.mi_paged_attn_prefill_takes_few(seqs, hkv, hq // hkv, q, keys))  # noqa: E731
    assert takes(1, 16, 8, 137, 144) and takes(16, 32, 8, 16, 2048) and takes(1, 8, 1, 256, 2304) and takes(40, 8, 8, 32, 2048)
    assert takes(1, 16, 8, 2048, 2048) and takes(2, 16, 8, 768, 1072) and takes(1, 32, 8, 576, 576) and takes(4, 16, 8, 288, 288) and takes(4, 8, 8, 576, 880)
    assert not takes(1, 8, 1, 2561, 2768) and not takes(1, 16, 1, 923, 928) and not takes(1, 32, 2, 914, 928) and not takes(1, 8, 1, 340, 2560)
    assert not takes(40, 32, 2, 14, 16) and not takes(2, 32, 8, 384, 688) and not takes(4, 8, 8, 1024, 1024) and not takes(1, 16, 8, 2049, 2064)
    assert not takes(1, 16, 8, 2048, 8192)   # (a table wider than the prompt: a prefix may lie in front of it)


def test_moe_tiles_refusals():
    """What mi_moe_tiles refuses before any launch: missing and misaligned operands, more tokens than pairs, sizes it does not take, and
    scratch that is a byte short."""
    from nanovllm import _C

    lib, EINVAL, EUNSUPPORTED, EWORKSPACE = _C.lib, -1, -2, -3
    pairs, E, H, I = 2400, 8, 1024, 512
    n = lib.mi_moe_tiles_bytes(pairs, E, I, H)
    assert n > 0 and lib.mi_moe_tiles_bytes(120, E, I, H) == 0 and lib.mi_moe_tiles_bytes(pairs, E, I + 8, H) == 0
    good = dict(x=4096, n_tokens=1200, gate_up=4096, down=4096, offsets=4096, pair_token=4096, pair_index=4096, act=4096, y=4096, pairs=pairs, n_experts=E,
                hidden=H, inter=I, scratch=4096, scratch_bytes=n - 1)   # (never read: the last refusal is the scratch's)
    call = lambda **k: lib.mi_moe_tiles(*{**good, **k}.values(), 0)  # noqa: E731
    codes = [call()]
    for name in ("x", "gate_up", "down", "act", "y", "scratch"):
        codes += [call(**{name: 0}), call(**{name: 4098})]
    for name in ("offsets", "pair_token", "pair_index"):
        codes.append(call(**{name: 0}))
    codes += [call(n_tokens=0), call(n_tokens=pairs + 1), call(pairs=120, n_tokens=60), call(inter=I + 8), call(scratch_bytes=0)]
    assert codes == [EWORKSPACE] + [EINVAL] * 15 + [EINVAL] * 2 + [EUNSUPPORTED] * 2 + [EWORKSPACE], codes


def test_delta_rule_by_blocks_rule():
    """From 32 rows of a sequence on, and half a row more for every sequence of the step; 0 floats of workspace elsewhere."""
    from nanovllm import _C

    blocks = lambda rows, seqs, most: _C.lib.mi_channel_delta_blocks_elems(rows, seqs, most, 8, 128) > 0  # noqa: E731
    assert blocks(33, 1, 33) and blocks(64 * 64, 64, 64) and blocks(160 + 255, 256, 160)
    assert not blocks(31, 1, 31) and not blocks(63 * 64, 64, 63) and not blocks(512, 256, 2) and not blocks(1, 1, 1)
