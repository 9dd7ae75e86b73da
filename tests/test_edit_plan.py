"""How a plain call's edits are put into passes (hd_edit_plan: the host's planning alone, no GPU)."""
import os

import pytest

from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(ROOT, "vkhashdag_amd", "libhashdag_amd.so")),
                                reason="library not built")


def spheres(centres, r, colored):
    return W.edits([W.edit(W.SPHERE_FILL, c, r2=r * r, color=0x4080C0 + k if colored else None, colored=colored)
                    for k, c in enumerate(centres)])


def test_edits_apart_share_passes_of_at_most_128():
    from vkhashdag_amd import capi
    e = spheres([(8 + 32 * (k % 16), 8 + 32 * (k // 16), 8) for k in range(256)], 3, True)
    cfg = small_cfg(1024, 9, 9, 2, 4)
    for n, want in ((2, [1, 1]), (3, [3]), (127, [127]), (128, [128]), (129, [128, 1]), (256, [128, 128])):
        assert capi.edit_plan(cfg, e[:n]) == want
    assert capi.edit_plan(cfg, W.edits([e[0], e[1], e[2], e[2], e[3], e[4]])) == [3, 3]


def test_one_node_level_has_no_chained_passes():
    """A pool of one level holds one leaf: edits apart from one another (one inside it, the others
    outside the grid) run one by one, for there are no inner nodes to keep versions of."""
    from vkhashdag_amd import capi
    e = spheres([(1, 1, 1), (40, 0, 0), (0, 80, 0), (0, 0, 120)], 1, False)
    assert capi.edit_plan(small_cfg(4, 2, 5, 2, 1), e) == [1, 1, 1, 1]
    assert capi.edit_plan(small_cfg(8, 2, 5, 2, 1), e) == [4]
