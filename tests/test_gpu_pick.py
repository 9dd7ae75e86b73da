"""Small inputs of a trace: rays in host memory (hd_traversal_host) against the same rays in device memory, and
views passed to the device as a kernel's arguments or by copies against each view traced alone."""
import ctypes as C
import threading

import numpy as np
import pytest

from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W

pytestmark = pytest.mark.gpu
RES = 128


@pytest.fixture(scope="module")
def pool():
    from vkhashdag_amd import capi
    p = capi.DevicePool(small_cfg(RES, 9, 9, 2, 3), heights=W.value_noise_heightmap(RES, 4, 5, 20, 100))
    p.edit(W.terrain_edit(RES, seed=3, skin=4))
    return p


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.random((n, 3), dtype=np.float32) + np.array([0, 0, 0.5], np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d[:, 2] = -np.abs(d[:, 2])
    return o, d


def _device(pool, o, d):
    from vkhashdag_amd import capi
    n = len(o)
    bo, bd, bout = capi.DeviceBuffer(o.nbytes), capi.DeviceBuffer(d.nbytes), capi.DeviceBuffer(n * 16)
    bo.upload(o)
    bd.upload(d)
    capi.check(capi.lib().hd_traversal(pool.h, pool.root, bo.ptr, bd.ptr, n, bout.ptr))
    return bout.download(np.float32, 4 * n).reshape(n, 4)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025])
def test_host_rays_equal_device_rays(pool, n):
    o, d = _rays(n, n)
    got, want = pool.traversal(o, d), _device(pool, o, d)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) and (n < 64 or want[:, 3].any())


def test_host_rays_refused_and_empty(pool):
    from vkhashdag_amd import capi
    o, d = _rays(1025, 1)
    out = np.zeros((1025, 4), np.float32)
    L = capi.lib()
    assert L.hd_traversal_host(pool.h, pool.root, o.ctypes.data, d.ctypes.data, 1025, out.ctypes.data) != 0
    assert L.hd_traversal_host(pool.h, pool.root, None, d.ctypes.data, 1, out.ctypes.data) != 0
    assert pool.traversal(o[:0], d[:0]).shape == (0, 4)


def test_host_rays_from_threads(pool):
    sets = [_rays(200 + k, 50 + k) for k in range(4)]
    want = [_device(pool, *s) for s in sets]
    got = [[None] * 20 for _ in sets]

    def go(k):
        for i in range(20):
            got[k][i] = pool.traversal(*sets[k])

    ts = [threading.Thread(target=go, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert all(np.array_equal(g, want[k]) for k in range(4) for g in got[k])


@pytest.mark.parametrize("beam", [False, True])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 40])
def test_views_equal_alone(pool, n, beam):
    from vkhashdag_amd import capi
    sizes = [(33 + 8 * (k % 5), 17 + 4 * (k % 7)) for k in range(n)]
    vbs = [W.orbit_view((64, 64, 50), 120.0, k, w, h, res=RES, lod=True) for k, (w, h) in enumerate(sizes)]
    views, at = (capi.hd_view * n)(), 0
    for k, (w, h) in enumerate(sizes):
        flags = capi.TRACE_SHADOW | (capi.TRACE_BEAM if beam and k % 2 == 0 else 0)
        views[k] = capi.make_view(vbs[k], w, h, flags, at)
        at += w * h
    for entry in ("hd_trace", "hd_trace_noalloc"):
        buf = capi.DeviceBuffer(at * 4)
        capi.check(getattr(capi.lib(), entry)(pool.h, pool.root, pool.color_root, C.cast(views, C.c_void_p), n, buf.ptr,
                                              None))
        got, at2 = buf.download(np.uint32, at), 0
        for k, (w, h) in enumerate(sizes):
            want = pool.render(vbs[k], w, h, shadow=True, beam=beam and k % 2 == 0)
            assert np.array_equal(got[at2:at2 + w * h], want), (entry, k)
            at2 += w * h
