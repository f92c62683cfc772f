"""The 2-column forms that mgbf_set_tile accepts (ti = 2 on the pass kinds 0, 1
and 2) are built: a kernel of 2 columns a lane for every half-width, kind of
taps, transfer stencil and band, by the compiler's report of the library."""
import json
import os
import re

import pytest

from standalone_mgbf_loc_amd import build as B

# template arguments H, TI, TAPS (0 box, 1 disc, 2 product), PRO, VHB, RES, QP
NAME = re.compile(r"radial_kernelILi(\d+)ELi(\d)ELi(\d)ELb(\d)ELi(\d)ELb(\d)ELb(\d)")


def test_every_accepted_two_column_form_is_built():
    if not os.path.exists(B.RESOURCES):
        pytest.skip("the library has not been built here")
    with open(B.RESOURCES) as f:
        built = {tuple(map(int, m.groups())) for m in map(NAME.search, json.load(f)) if m}
    assert built
    for four in built:
        h, ti, taps, pro, vhb, res, qp = four
        if ti == 4 and not res:
            assert (h, 2, taps, pro, vhb, res, qp) in built, four
