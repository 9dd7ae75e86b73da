"""Plain calls whose edits share passes (versions of the nodes near the root), at the edges of what such a
pass takes: pools of one and two node levels."""
import pytest

import _oracle as O
from test_edit_plan import spheres
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [4, 8])
def test_few_node_levels(res):
    from vkhashdag_amd import capi
    print(f"{res}^3, edits inside and outside the grid", flush=True)
    cfg = small_cfg(res, 2, 5, 2, 1)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    for k in range(3):
        e = spheres([(1 + k, 1, 1), (40, 0, 0), (res - 1, res - 1, res - 1 - k), (0, 80, 0), (0, 0, 120)], 1 + k % 2, False)
        dev.edit(e)
        ora.edit(e)
        assert_same_pool(dev, ora, f"call {k}")
    assert dev.stats().overflow == 0
