"""Color jobs rebuilt segment by segment: chunks of 64, 512 and 4096 voxels (few or all threads of the workgroup
hold voxels), plain and weighted colors mixed inside a segment, chunks staged or encoded in place, against the
CPU oracle after every edit."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_colors import weighted_edits
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("staging", ["", "16"])
@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("depth", [2, 3, 4])
def test_jobs_bit_exact(depth, keep, staging, monkeypatch):
    from vkhashdag_amd import capi
    if staging:
        monkeypatch.setenv("HD_EDIT_STAGING_WORDS", staging)
    cfg = small_cfg(64, 8, 6, 2, depth, keep_history=keep)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    e = weighted_edits(20, 64, 40 + depth)
    # single voxels and thin slabs inside one leaf: segments of up to 16 colors, weighted and not
    rng = np.random.default_rng(depth)
    fine = []
    for k in range(40):
        lo = tuple(int(v) for v in rng.integers(16, 32, 3))
        hi = tuple(int(v + rng.integers(1, 5)) for v in lo)
        r = W.edit(W.AABB_PAINT if k % 3 else W.AABB_FILL, lo, hi, color=int(rng.integers(1 << 24)))
        if k % 4 == 1:
            r["bpw"] = 1 + k % 3
            r["weight"] = int(rng.integers(0, 2 << (k % 3)))
        fine.append(r)
    e = W.edits(list(e[:10]) + fine + list(e[10:]))
    for i in range(len(e)):
        dev.edit(e[i:i + 1])
        ora.edit(e[i:i + 1])
        assert_same_pool(dev, ora, f"depth {depth} keep {keep} edit {i}")
