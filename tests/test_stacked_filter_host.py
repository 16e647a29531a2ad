"""The stacked gates filter of a ConvGRU: a captured step holds the addresses of one of its two column orders."""
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
