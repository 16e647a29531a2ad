"""The stacked gates conv of a ConvGRU on the host: its filter, of which a captured step holds one of two column orders, and its form."""
import gc
import weakref

import pytest
import torch

from maskedincrementeval_amd import ops
from maskedincrementeval_amd.evflownet_incr import ConvGRUIncr


@pytest.mark.parametrize("first", [False, True])
def test_a_column_order_outlives_a_call_in_the_other(first):
    cell = ConvGRUIncr(16, 16, 3)
    kept = weakref.ref(cell._stacked_filter(first))
    cell._stacked_filter(not first)
    gc.collect()
    assert kept() is not None and cell._stacked_filter(first) is kept()
    # the same columns, each in its order; a weight that changes is seen by both
    with torch.no_grad():
        cell.out_gate.weight.mul_(2)
    want = torch.cat((cell.update_gate.weight, cell.out_gate.weight), 0).detach().permute(1, 2, 3, 0)
    assert torch.equal(cell._stacked_filter(False).plain, want)
    assert torch.equal(cell._stacked_filter(True).plain, want[..., ops.gru_interleave_index(16)])
    gc.collect()
    assert kept() is None


def test_where_the_gates_of_many_channels_stay_two_calls():
    f32, bf16 = torch.float32, torch.bfloat16
    for hid, tiles, line in ((64, 16, 1024), (32, 32, 1024), (64, 17, 512), (256, 8, 512)):      # slabs 128, 128, 136, 256
        assert ops.conv_gru_takes(line, 2 * line, hid, f32, tiles) and not ops.conv_gru_takes(line + 64, 2 * line, hid, f32, tiles)
        assert ops.conv_gru_takes(line + 64, 2 * line, hid, bf16, tiles) and ops.conv_gru_takes(line + 64, 2 * line, hid, f32)
    assert ops.conv_gru_takes(2048, 2048, 256, f32, 9)                                           # not split: 288
