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


def assert_same_devices(a, b, where):
    from vkhashdag_amd import capi
    assert (a.root, a.color_root) == (b.root, b.color_root), where
    assert a.stats().overflow == b.stats().overflow, where
    assert all(np.array_equal(x, y) for x, y in zip(a.live_words(), b.live_words())), where
    # (the counts go on past the capacity, and what did not fit leaves its words unwritten: the colors are compared)
    counts = [(p.stats().color_nodes, p.stats().color_leaf_words) for p in (a, b)]
    assert counts[0] == counts[1], where
    nodes, words = min(counts[0][0], a.cfg.color_node_capacity), min(counts[0][1], a.cfg.color_leaf_capacity)
    vox = np.random.default_rng(1).integers(0, 1 << a.cfg.voxel_level, (20000, 3)).astype(np.uint32)
    vox[:, 2] = 90 + vox[:, 2] % 32
    got = []
    for p in (a, b):
        cn, cl = np.zeros(max(nodes, 1) * 8, np.uint32), np.zeros(max(words, 1), np.uint32)
        capi.check(capi.lib().hd_pool_read_color_nodes(p.h, 0, nodes, cn.ctypes.data))
        capi.check(capi.lib().hd_pool_read_color_leaves(p.h, 0, words, cl.ctypes.data))
        got.append(O.color_fetch(cn, cl, p.color_root, p.cfg.voxel_level, p.cfg.color_leaf_level, vox))
    assert np.array_equal(*got), where


# the calls below take 184 to 259 color nodes and 9800 color leaf words
@pytest.mark.parametrize("nodes,words", [(1 << 16, 5000), (220, 1 << 20), (1 << 16, 1 << 20)])
def test_color_pool_runs_out(nodes, words):
    """Edits of one call where the color nodes or leaves end: as the same edits one call each."""
    from vkhashdag_amd import capi
    res = 256
    print(f"{nodes} color nodes, {words} color leaf words", flush=True)
    cfg = small_cfg(res, 9, 9, 2, 4, color_node_capacity=nodes, color_leaf_capacity=words)
    a, b = capi.DevicePool(cfg), capi.DevicePool(cfg)
    e = W.edits([W.edit(W.AABB_FILL, (0, 0, 0), (res, res, 100), color=0x305070)])
    for k in range(5):
        a.edit(e)
        for i in range(len(e)):
            b.edit(e[i:i + 1])
        assert_same_devices(a, b, f"call {k}")
        e = spheres([(16 + 48 * i + k, 16 + 48 * j, 100 + 3 * k) for i in range(5) for j in range(5)], 6, True)
    assert (a.stats().overflow == 0) == (nodes == words >> 4)


def test_color_words_of_more_than_rgb8():
    """Words with bits above the 24 of RGB8, and weights of no bits: as the same edits one call each."""
    from vkhashdag_amd import capi
    res = 256
    print("color words of 32 bits", flush=True)
    cfg = small_cfg(res, 9, 9, 2, 4)
    a, b = capi.DevicePool(cfg), capi.DevicePool(cfg)
    rng = np.random.default_rng(3)
    palette = np.array([0x305070, 0xFF305070, 0x12345678, 0x00305071], np.uint32)
    e = W.edits([W.edit(W.AABB_FILL, (0, 0, 0), (res, res, 100), color=0x111111)])
    for k in range(5):
        a.edit(e)
        assert k != 1 or a.edit_passes()[0] < len(e)
        for i in range(len(e)):
            b.edit(e[i:i + 1])
        assert_same_devices(a, b, f"call {k}")
        e = spheres([(24 + 48 * i, 24 + 48 * j, 100) for i in range(5) for j in range(5)], 7 + k % 2, True)
        e["colors"] = palette[rng.integers(0, 4, len(e))]
        e["weight"] = rng.integers(0, 2, len(e))
        e["kind"] = rng.choice([W.SPHERE_FILL, W.SPHERE_PAINT], len(e))
