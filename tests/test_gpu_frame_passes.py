"""A frame replays as many passes as its edits need: frames of 0 to max_passes dependent groups, in mixed order,
queued and relaunched, against batched edits of the same lists."""
import numpy as np
import pytest

from test_gpu_async import assert_equivalent_device_pools
from test_gpu_frame import _terrain, _views
from vkhashdag_amd import workloads as W

pytestmark = pytest.mark.gpu


def _nested(res, n, seed):
    """n edits that all overlap: n groups, one pass each."""
    rng = np.random.default_rng(seed)
    c = tuple(int(v) for v in rng.integers(res // 4, res * 3 // 4, 3))
    return W.edits([W.edit(W.SPHERE_DIG if k % 2 else W.SPHERE_FILL, c, r2=(12 - k) ** 2,
                           color=None if k % 2 else int(rng.integers(1 << 24))) for k in range(n)]) if n else []


@pytest.mark.parametrize("max_passes,gc", [(1, False), (2, False), (3, True), (5, False), (8, True)])
def test_frames_of_every_pass_count(max_passes, gc):
    from vkhashdag_amd import capi
    res = 128
    cfg, _, (a, b) = _terrain(capi, res, seed=4)
    f = capi.Frame(a, max_edits=4, max_passes=max_passes, max_radius=16, n_views=2, max_width=64, max_height=48, gc=gc)
    counts = [0, max_passes, 1, 0, max_passes - 1, *range(max_passes + 1), max_passes]
    for k, n in enumerate(counts):
        e = _nested(res, n, 60 + k)
        f.set(e, _views(res, k))
        f.launch()
        if k % 3 == 1:
            f.launch()  # the same edits again, before anything is read back
        f.wait()
        for _ in range(2 if k % 3 == 1 else 1):
            for i in range(n):
                b.edit(e[i:i + 1])
        if gc:
            b.gc([])
        assert_equivalent_device_pools(a, b, cfg, f"frame {k}, {n} passes")
        for (vb, w, h, _), img in zip(_views(res, k), f.images()):
            assert np.array_equal(img, a.render(vb, w, h, shadow=True)), f"frame {k}: view differs"
    f.close()
