"""The mesh calls where their (face, cell) pairs outnumber what 32-bit list
starts can hold: 2^31 pairs or more are refused with CVT_ERR_CAPACITY before
any list is filled, the outputs untouched, and the next call is right.  (The
starts of that many pairs wrap, to values that look like small lists.)"""
import numpy as np
import pytest

from test_gpu_locate import check as check_locate
from test_oracle import jittered_mesh

pytestmark = pytest.mark.gpu

CAPACITY = -5


def covering(num, extent):
    """num triangles (distinct, not thin) whose boxes cover [0, extent]^2"""
    t = np.arange(num) * (extent / num)
    p = np.stack([np.stack([0 * t - extent, 0 * t - extent], 1),
                  np.stack([0 * t + 3 * extent, t - extent], 1),
                  np.stack([t - extent, 0 * t + 3 * extent], 1)], 1)
    return p.reshape(-1, 2), np.arange(3 * num, dtype=np.int32).reshape(-1, 3)


def refused(call):
    from cvtamd import CvtError
    with pytest.raises(CvtError) as e:
        call()
    assert e.value.status == CAPACITY, e.value


# 1024^2 tiles a triangle: 2^31 pairs exactly, and 2^32 + 2^20, whose wrapped total is small
@pytest.mark.parametrize("num", [2048, 4097])
def test_raster_refuses(gpu, orc, num):
    import torch
    from cvtamd import compat
    n = 16384
    pts, tri = covering(num, float(n))
    w = np.ones(len(pts))
    out = torch.full((n, n), 7.0, dtype=torch.float32, device="cuda")
    print(f"raster {num} x {n}^2", flush=True)
    refused(lambda: compat.rasterize(pts, w, tri, 1.0, n, out=out))
    assert bool((out == 7).all())
    uv, mt = jittered_mesh(12, 3)
    wm = np.random.default_rng(4).random(len(uv))
    assert np.array_equal(compat.rasterize(uv, wm, mt, 0.1, 200), orc.raster(uv, wm, mt, 0.1, 200))


def test_raster_noalloc_refuses(gpu):
    import ctypes as C
    import torch
    from cvtamd._lib import call
    n, num = 4096, 32768 + 64                      # 256^2 tiles: 2^31 + 2^22 pairs
    pts, tri = covering(num, float(n))
    d = [torch.from_numpy(a).cuda() for a in (pts, np.ones(len(pts)), tri)]
    out = torch.full((n, n), 7.0, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    ptr = lambda t: C.c_void_p(t.data_ptr())
    print("raster_noalloc", flush=True)
    refused(lambda: call("cvt_rasterize_noalloc", ptr(d[0]), ptr(d[1]), len(pts), ptr(d[2]), num,
                         ptr(out), 1.0, n))
    assert bool((out == 7).all())


def test_locate_refuses(gpu):
    import torch
    from cvtamd import recover
    num = 65600                                    # 182^2 bins: 1.01 * 2^31 pairs
    t = np.linspace(0.0, 1e-3, num)
    # every face's box meets every bin
    p = np.stack([np.stack([t, t], 1), np.stack([1.0 - 0 * t, t], 1),
                  np.stack([t, 1.0 - 0 * t], 1)], 1).reshape(-1, 2)
    tri = np.arange(3 * num, dtype=np.int32).reshape(-1, 3)
    q = torch.rand(100, 2, dtype=torch.float64, device="cuda")
    out = (torch.full((100,), 7, dtype=torch.int32, device="cuda"),
           torch.full((100, 3), 7.0, dtype=torch.float64, device="cuda"))
    print("locate", flush=True)
    refused(lambda: recover.locate_points(p, tri, q, out=out))
    for o in out:
        assert bool((o == 7).all())
    uv, mt = jittered_mesh(12, 3)
    check_locate(uv, mt, np.random.default_rng(5).uniform(0, 11, (500, 2)),
                 np.stack([uv[:, 0], uv[:, 1], uv[:, 0]], 1))
