"""CPU replay of the training attention's launch order (fa_block_order of nanochat_amd/csrc/flash_attn.hip): an XCD's
second 32 work-groups, or as many as there are in whole rows of eight, are taken in reverse. For every number of
work-groups each place of the linear order is taken once, and the counts that tests/test_gpu_flash_attn.py runs reach a
full, a part-filled and no reversed round. The constants are read from the source."""
import re

import pytest

from nanochat_amd import native

SOURCE = (native.CSRC / "flash_attn.hip").read_text()
XCDS, XCD_CUS = map(int, re.search(r"FA_XCDS = (\d+), FA_XCD_CUS = (\d+)", SOURCE).groups())


def order(everything):
    """The place in launch order that each work-group L takes."""
    end = min(2 * XCD_CUS, everything // XCDS)
    places = []
    for L in range(everything):
        n = L // XCDS
        places.append((XCD_CUS + end - 1 - n) * XCDS + L % XCDS if XCD_CUS <= n < end else L)
    return places


def test_the_replay_is_the_kernels_rule():
    body = " ".join(re.search(r"FaBlock fa_block_order\(\) \{(.*?)\n\}", SOURCE, re.S).group(1).split())
    assert "end = min(2 * FA_XCD_CUS, all / FA_XCDS)" in body
    assert "if (n >= FA_XCD_CUS && n < end) L = (FA_XCD_CUS + end - 1 - n) * FA_XCDS + L % FA_XCDS;" in body


def test_every_place_is_taken_once():
    for everything in range(1, 2001):
        assert sorted(order(everything)) == list(range(everything)), everything


@pytest.mark.parametrize("everything,reversed_rows", [(1, 0), (256, 0), (270, 1), (272, 2), (369, 14), (511, 31), (512, 32),
                                                      (540, 32), (6144, 32)])
def test_reversed_rows(everything, reversed_rows):
    """Rows of eight in the reversed second round; one row in reverse is that row."""
    places = order(everything)
    moved = [L for L in range(everything) if places[L] != L]
    lo, hi = XCDS * XCD_CUS, XCDS * (XCD_CUS + reversed_rows)
    assert all(lo <= L < hi for L in moved)
    assert len(moved) == (reversed_rows // 2 * 2 * XCDS)
    assert all(places[L] == lo + hi - XCDS - L + 2 * (L % XCDS) for L in moved)
