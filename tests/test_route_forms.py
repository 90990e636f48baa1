"""The forms that calls take by rules on their sizes, checked on the host through
the route query (its grids are those of 256 compute units where no device is
current): calls on either side of a rule, each measured both ways."""
import pytest
import torch

import hsdpa

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="a device's own compute units would count")


@pytest.mark.parametrize("heads,kv_heads,rows,past,sink,shares", [
    # us in equal shares against the other form
    (16, 2, 3238, 0, False, False),      # 193, paired 147: nine short row groups in the first share
    (16, 4, 3435, 0, False, False),      # 186, paired 150
    (32, 4, 1469, 0, False, False),      # 112, one launch 97
    (16, 2, 1779, 0, False, False),      # 90, split in two 76
    (8, 2, 1718, 336, False, False),     # 61, split in four 56: two pieces a share of eight tiles
    (32, 4, 138, 4521, True, False),     # 71, split in eight 65: 14 maxima a row group
    (16, 2, 2122, 5515, False, True),    # 275, one launch 452
    (8, 2, 2912, 1056, False, True),     # 102, split in two 148
    (12, 4, 2887, 1667, False, True),    # 165, paired 231
    (24, 12, 811, 5143, True, True),     # 162, split in two 221
])
def test_equal_shares(heads, kv_heads, rows, past, sink, shares):
    plan = hsdpa.Plan(heads, heads // kv_heads, 128, rows + past, sink=sink)
    r = plan.route(rows, past)
    assert (r["splits"] == 0) == shares, r
