"""Column fills on the sync-free pipeline: its per-level entry counts come from the heightfield's min / max
pyramid, so heightfields at the counts' edges (empty, full, flat, steps on and beside node faces, ragged
rectangles, skins deeper than the terrain) against the CPU oracle, with and without colors."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W

pytestmark = pytest.mark.gpu
RES = 128


def _heights(kind, res):
    y, x = np.mgrid[0:res, 0:res].astype(np.uint32)
    if kind == "noise":
        return W.value_noise_heightmap(res, 4, 3, res // 6, res * 3 // 4)
    if kind == "steps":  # faces of 4-, 8-, 16-voxel nodes and one voxel to either side
        return np.take(np.array([0, 1, 15, 16, 17, 31, 32, 33, 64, 127, 128], np.uint32), (x // 8 + 3 * (y // 8)) % 11)
    if kind == "spikes":
        return np.where((x * 7 + y * 13) % 61 == 0, res, 3).astype(np.uint32)
    return np.full((res, res), {"empty": 0, "one": 1, "flat": 48, "full": res}[kind], np.uint32)


RECTS = [((0, 0), (RES, RES)), ((5, 17), (94, 101)), ((64, 0), (128, 64)), ((3, 3), (4, 4)), ((9, 9), (9, 40))]


@pytest.mark.parametrize("colored", [False, True])
@pytest.mark.parametrize("kind", ["noise", "steps", "spikes", "empty", "one", "flat", "full"])
def test_column_fill_vs_oracle(kind, colored):
    from vkhashdag_amd import capi
    h = np.ascontiguousarray(_heights(kind, RES))
    cfg = small_cfg(RES, 9, 9, 2, 3)
    for lo, hi in RECTS:
        for skin in (0, 3, 200):
            print(f"{kind} colored={colored} rect {lo} {hi} skin {skin}", flush=True)
            dev, ora = capi.DevicePool(cfg, heights=h), O.OraclePool(cfg, heights=h)
            e = W.edits([W.edit(W.SPHERE_FILL, (60, 60, 40), r2=900, color=0x3060A0 if colored else None,
                                colored=colored),
                         W.terrain_edit(RES, seed=2, skin=skin, lo=lo, hi=hi, colored=colored),
                         W.terrain_edit(RES, seed=2, skin=skin, colored=colored)])
            for i in range(len(e)):
                dev.edit(e[i:i + 1])
                ora.edit(e[i:i + 1])
                assert_same_pool(dev, ora, f"edit {i}")


@pytest.mark.parametrize("res", [64, 256, 1024])
def test_column_fill_equals_synchronized(res, monkeypatch):
    from vkhashdag_amd import capi
    cfg = small_cfg(res, 12, 9, 3, 4)
    heights = W.value_noise_heightmap(res, 5, 8, res // 8, res * 3 // 4)
    got = []
    for path in ("", "sync"):
        monkeypatch.setenv("HD_EDIT_PATH", path)
        dev = capi.DevicePool(cfg, heights=heights)
        dev.edit(W.terrain_edit(res, seed=1, skin=6))
        dev.edit(W.edits([W.terrain_edit(res, seed=9, skin=2, lo=(res // 3, 1), hi=(res - 5, res // 2))]))
        got.append((dev.root, dev.color_root, dev.live_words()[1], dev.color_leaves(), dev.stats().overflow))
    assert got[0][:2] == got[1][:2] and got[0][4] == got[1][4] == 0
    assert np.array_equal(got[0][2], got[1][2]) and np.array_equal(got[0][3], got[1][3])
