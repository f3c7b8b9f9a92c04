"""Which calls the medium-row products (exl3_dgemm) take, decided on the host -- no GPU."""
import ctypes
import pytest


def _block(hidden, inter, experts):
    from exllamav3_amd.moe_path import SyntheticEXL3MoE
    b = SyntheticEXL3MoE.__new__(SyntheticEXL3MoE)
    b.hidden, b.inter, b.E = hidden, inter, experts
    return b


@pytest.mark.parametrize("hidden,inter,experts,tokens,top,packed", [
    (4096, 14336, 8, 1100, 2, True), (4096, 14336, 8, 2560, 2, True), (4096, 14336, 8, 2561, 2, False),             # rows per expert
    (7168, 2048, 256, 18000, 8, True), (7168, 2048, 256, 19000, 8, False), (2048, 7168, 256, 19000, 8, False),     # scratch of the gate / up and of the down product
    (8192, 1024, 512, 40000, 8, False), (2048, 768, 128, 10000, 8, True)])
def test_expert_block_leaves_the_packed_route_where_its_scratch_ends(hidden, inter, experts, tokens, top, packed):
    assert _block(hidden, inter, experts)._on_packed_weights(tokens * top) == packed


@pytest.mark.parametrize("groups,k", [(8, 14336), (256, 7168), (100, 2048)])
def test_rule_and_entry_point_agree_on_the_largest_call(groups, k):
    """The last row count that dgemm_grouped_fits allows is the last one for which the C entry does not name its limit (arguments are checked before anything is launched)."""
    from exllamav3_amd import _lib, ext
    lo, hi = 1, 1 << 20
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if ext.dgemm_grouped_fits(mid, groups, k) else (lo, mid)
    l = _lib.lib()

    def refused(rows):
        tile = ext._group_tile(rows, groups)
        need = l.exl3_dgemm_grouped_xh_rows(rows, tile)
        # (an output pointer off its alignment: a call within the limit ends at that check, the next one behind the limit's)
        rc = l.exl3_dgemm_grouped(16, None, k, None, 16, 16, need, 16, 16, 16, groups, (ctypes.c_void_p * 1)(8), 128, 128, 1, 1, rows, tile, k, 4, 2, None)
        text = l.exl3_last_error()
        assert rc < 0 and (b"below 2 GiB" in text or b"aligned outputs" in text), text
        return b"below 2 GiB" in text
    assert not refused(lo) and refused(hi)


def test_segments_of_a_layer_without_weights():
    """The cut of a prompt into segments is asked of a layer by its sizes alone (the benchmark of the mixer families does)."""
    import torch
    from exllamav3_amd.modules import GatedLinearAttention
    from exllamav3_amd.state_cache import StepBatch
    none = torch.zeros(1, dtype=torch.int32)
    step = lambda rows: StepBatch(rows, 1, False, rows, None, none, none, none, none, none, none)
    for dim, least in ((64, 48), (128, 48), (96, 256)):
        layer = GatedLinearAttention(2048, 16, dim, 128, 16.0, 1e-5)
        assert layer.segments(step(least - 1)) is None
        segs, length = layer.segments(step(4096))
        assert segs >= 2 and segs * length >= 4096 and (dim == 96 or length % 16 == 0)
