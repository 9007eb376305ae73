"""Decode launch lists of many rows with short ones among them."""
import numpy as np
import pytest

from test_abi import GROUPS, W, _check_decode_schedule, _schedule, lib  # noqa: F401  (lib: fixture)


@pytest.mark.parametrize("rows,lo,hi,seed", [(200, 100, 3000, 1), (256, 16, 8000, 2), (150, 16, 2000, 3), (255, 1, 400, 4)])
def test_no_second_round_of_work_groups(lib, rows, lo, hi, seed):  # noqa: F811
    """Work-groups that close early (W short segments) make more of them than
    a device-full; the planner then weighs the second round, and the last
    work-group does not end long after an even share."""
    k = np.random.default_rng(seed).integers(lo, hi + 1, rows)
    dec, _, merge, ws, qs = _schedule(lib, [1] * rows, k, k - 1)
    loads = _check_decode_schedule(dec, merge, ws, qs, W, dict(enumerate(k.tolist())), 8)
    even = sum(-(-int(x) // 16) for x in k) * 8 / GROUPS
    ends = [0] * GROUPS  # work-groups taken in order by the resident ones
    for x in loads:
        ends.sort()
        ends[0] += x
    assert max(ends) <= even * 1.1 + 14  # 14 slices: what a merge launch costs, and one more
