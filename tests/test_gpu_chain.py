"""Several edits of one plain call in one pass (chained passes): the pool words, bucket counters, roots,
color nodes and color leaves equal the oracle's sequential edits (= the reference's Edit applied to each
in turn), whatever the edits share: nodes near the root, emptied or newly filled ones, colors."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W

pytestmark = pytest.mark.gpu
KINDS = [W.SPHERE_FILL, W.SPHERE_DIG, W.SPHERE_PAINT, W.AABB_FILL, W.AABB_DIG, W.AABB_PAINT]


def small_edits(n, res, seed, colored, rmax, palette, kinds=KINDS):
    """Small edits all over the grid: spheres and boxes, colors from a palette (few: many are equal)."""
    rng = np.random.default_rng(seed)
    colors = rng.integers(0, 1 << 24, palette)
    out = []
    for _ in range(n):
        k = kinds[int(rng.integers(len(kinds)))]
        c = rng.integers(-2 if k < 3 else 0, res + 3, 3).clip(0)
        r = int(rng.integers(0, rmax + 1))
        col = int(colors[int(rng.integers(palette))])
        dig = k in (W.SPHERE_DIG, W.AABB_DIG)
        if k in (W.SPHERE_FILL, W.SPHERE_DIG, W.SPHERE_PAINT):
            out.append(W.edit(k, tuple(int(v) for v in c), r2=r * r + int(rng.integers(0, 2)), color=None if dig else col,
                              colored=colored and not dig))
        else:
            lo = tuple(int(v) for v in (c - r).clip(0))
            out.append(W.edit(k, lo, tuple(int(v) for v in c + rng.integers(0, r + 2, 3)), color=None if dig else col,
                              colored=colored and not dig))
    return W.edits(out)


@pytest.mark.parametrize("colored", [True, False])
@pytest.mark.parametrize("res,rmax,palette,seed", [(64, 2, 40, 1), (64, 5, 1, 2), (128, 4, 3, 3), (256, 9, 1, 4),
                                                   (256, 12, 60, 5), (512, 20, 2, 6)])
def test_chained_edits_bit_exact(res, rmax, palette, seed, colored):
    from vkhashdag_amd import capi
    print(f"chain {res} r<={rmax} palette {palette} colored {colored}", flush=True)
    h = W.value_noise_heightmap(res, 4, seed, res // 5, res * 3 // 4)
    cfg = small_cfg(res, 9, 9, 2, 3 if seed % 2 else 4, )
    kinds = KINDS if colored else KINDS[:2] + KINDS[3:5]
    dev, ora = capi.DevicePool(cfg, heights=h), O.OraclePool(cfg, heights=h)
    base = W.edits([W.terrain_edit(res, seed=3, skin=6, colored=colored)])
    for p in (dev, ora):
        p.edit(base)
    for k in range(4):
        e = small_edits(60, res, 10 * seed + k, colored, rmax, palette, kinds)
        if k % 2:  # on the surface, where the world's own nodes are
            xy = e["p0"][:, :2].clip(0, res - 1)
            z = h[xy[:, 1], xy[:, 0]]
            e["p1"][:, 2] = np.where(e["kind"] >= 3, z + (e["p1"][:, 2] - e["p0"][:, 2].astype(np.int64)).clip(0), 0)
            e["p0"][:, 2] = z
        dev.edit(e)
        ora.edit(e)
        assert_same_pool(dev, ora, f"call {k}")


@pytest.mark.parametrize("colored", [True, False])
def test_chained_edits_from_an_empty_pool(colored):
    """The first edits of a pool: a null root, nodes that earlier edits of the pass filled or emptied."""
    from vkhashdag_amd import capi
    cfg = small_cfg(128, 6, 5, 4, 4)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    kinds = KINDS if colored else KINDS[:2] + KINDS[3:5]
    for k in range(6):
        e = small_edits(25, 128, 50 + k, colored, 3 + 2 * k, 1 + k, kinds)
        dev.edit(e)
        ora.edit(e)
        assert_same_pool(dev, ora, f"call {k}")


def test_chained_edits_in_full_buckets():
    """Buckets so small that appends fail (the reference keeps the old pointer): the same fallbacks."""
    from vkhashdag_amd import capi
    cfg = small_cfg(128, 3, 5, 1, 4)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    for k in range(5):
        e = small_edits(40, 128, 80 + k, False, 6, 1, KINDS[:2] + KINDS[3:5])
        dev.edit(e)
        ora.edit(e)
        assert_same_pool(dev, ora, f"call {k}")
    assert ora.overflows() > 0
