"""New nodes of a level's buckets around the walker's limits (1 to 4 by one thread, 5 to 64 by a wavefront, more by
a chain): few buckets and passes of growing size, every pool word against the CPU oracle."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg
from vkhashdag_amd import capi
from vkhashdag_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [3, 6, 9, 11])
@pytest.mark.parametrize("colored", [False, True])
def test_walks_of_every_list_length(bits, colored):
    res = 256
    cfg = small_cfg(res, bits, 9, 5, 3)
    h = W.value_noise_heightmap(res, 6, bits, 30, 200)
    dev, ora = capi.DevicePool(cfg, heights=h), O.OraclePool(cfg, heights=h)
    rng = np.random.default_rng(bits)
    e = [W.edit(W.SPHERE_FILL if k % 2 == 0 else W.SPHERE_DIG, tuple(int(v) for v in rng.integers(40, 216, 3)),
                r2=int(r) ** 2, color=int(rng.integers(1 << 24)) if colored and k % 2 == 0 else None,
                colored=colored and k % 2 == 0) for k, r in enumerate([3, 5, 8, 12, 18, 26, 36, 48])]
    e.append(W.terrain_edit(res, seed=1, skin=4, colored=colored))
    for i in range(len(e)):
        dev.edit(W.edits(e[i:i + 1]))
        ora.edit(W.edits(e[i:i + 1]))
        assert_same_pool(dev, ora, f"bits {bits} edit {i}")
