"""Plain calls whose edits share passes (versions of the nodes near the root), at the edges of what such a
pass takes: pools of one and two node levels, edits that meet in empty space, runs of its most edits,
color leaves that keep their history."""
import numpy as np
import pytest

import _oracle as O
from test_edit_plan import spheres
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W

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


@pytest.mark.parametrize("name,step,grid", [("row", 32, (28, 1, 1)), ("sheet", 48, (16, 16, 1)), ("lattice", 40, (6, 6, 6)),
                                            ("three", 40, (3, 1, 1))])
def test_colored_edits_that_meet_in_empty_space(name, step, grid):
    """Fills in the air of a world: no two share a color leaf, but many share empty nodes above it. Most runs
    are found out after their top-down, and the call takes few passes more than it has edits."""
    from vkhashdag_amd import capi
    res = 1024
    print(f"{name} of {grid} fills, {step} apart", flush=True)
    cfg = small_cfg(res, 9, 9, 2, 4)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    ground = W.edits([W.edit(W.AABB_FILL, (0, 0, 0), (res, res, 600), color=0x305070)])
    centres = [(40 + step * x, 40 + step * y, 700 + step * z) for z in range(grid[2]) for y in range(grid[1])
               for x in range(grid[0])]
    for e in (ground, spheres(centres, 6, True), spheres([(x + 5, y, z) for x, y, z in centres], 6, True)):
        dev.edit(e)
        ora.edit(e)
        applied, left, cut = dev.edit_passes()
        assert_same_pool(dev, ora, name)
        n = len(e)
        assert applied + left + cut <= n + max(1, n // 8), (n, applied, left, cut)


@pytest.mark.parametrize("colored", [True, False])
@pytest.mark.parametrize("n", [127, 128, 129, 300])
def test_runs_of_the_most_edits(n, colored):
    from vkhashdag_amd import capi
    res = 512
    print(f"{n} edits apart, colored {colored}", flush=True)
    cfg = small_cfg(res, 9, 9, 2, 4)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    ground = W.edits([W.edit(W.AABB_FILL, (0, 0, 0), (res, res, res), color=0x305070, colored=colored)])
    rng = np.random.default_rng(n)
    order = rng.permutation(16 * 16 * 4)[:n]
    e = spheres([(12 + 32 * (k % 16), 12 + 32 * (k // 16 % 16), 60 + 96 * (k // 256)) for k in order], 4, colored)
    e["kind"][::3] = W.SPHERE_DIG
    e["colored"][::3] = 0
    for part in (ground, e):
        dev.edit(part)
        ora.edit(part)
        assert_same_pool(dev, ora, f"{n} edits")
    applied, left, cut = dev.edit_passes()
    assert (left, cut) == (0, 0) and applied <= (n + 127) // 128 + 1


@pytest.mark.parametrize("history", [True, False])
def test_color_leaves_in_place_or_kept(history):
    """The same places again and again: color leaves that fit are written in place, unless the pool keeps them."""
    from vkhashdag_amd import capi
    res = 256
    print(f"keep_history {history}", flush=True)
    cfg = small_cfg(res, 9, 9, 2, 4, keep_history=history)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    ground = W.edits([W.edit(W.AABB_FILL, (0, 0, 0), (res, res, 100), color=0x305070)])
    dev.edit(ground)
    ora.edit(ground)
    words = []
    for k in range(4):
        e = spheres([(16 + 48 * i, 16 + 48 * j, 100) for i in range(5) for j in range(5)], 5 + k % 2, True)
        e["kind"][k::4] = W.SPHERE_PAINT
        dev.edit(e)
        ora.edit(e)
        assert_same_pool(dev, ora, f"call {k}")
        assert dev.edit_passes()[0] < len(e)
        words.append(dev.stats().color_leaf_words)
    assert not history or words == sorted(set(words))  # nothing in place: it grows with every call
