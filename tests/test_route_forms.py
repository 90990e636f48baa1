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


@pytest.mark.parametrize("heads,kv_heads,dim,rows,past,cap,groups", [
    # us over all groups against a workgroup per group; the cache's capacity
    (16, 2, 256, 14, 7982, 40000, False),     # 33.6, 28.7: seven groups of 4 tiles in turn
    (32, 4, 256, 12, 4019, 40000, False),     # 34.7, 30.4
    (16, 2, 256, 14, 27312, 40000, True),     # 48.1, 66.0
    (128, 16, 256, 8, 6007, 40000, True),     # 56.4, 81.8
    (32, 8, 128, 16, 5147, 40000, False),     # 31.0, 29.8: a chunk of 8 tiles for 6
    (128, 16, 128, 6, 6130, 40000, True),     # 37.0, 51.5
    # workspaces with fewer workgroups: kept within 32 MiB, or for a short cache
    (16, 2, 256, 12, 5757, 5769, False),      # 30.6, 28.8
    (16, 2, 256, 16, 11984, 12000, False),
    (128, 16, 256, 11, 610, 621, True),       # 47.4, 48.7; 60 in runs per group
    (32, 8, 128, 16, 12379, 12395, False),    # 59.2, 48.1
])
def test_all_groups(heads, kv_heads, dim, rows, past, cap, groups):
    r = hsdpa.Plan(heads, heads // kv_heads, dim, cap, max_rows=rows).route(rows, past)
    assert (r["main"], r["splits"] == 0) == ("few_rows", groups), r
