"""The mesh calls (cvt_rasterize, cvt_locate_points, cvt_vertex_weights) where
their lists outgrow the room they first get, at the sizes where the scan of
the counts changes, with arguments in device memory used in place, with
outputs that meet an input, and from several threads.  Bar: bit-exact."""
import ctypes as C
import threading

import numpy as np
import pytest

from test_gpu_locate import check as check_locate, queries
from test_oracle import jittered_mesh

pytestmark = pytest.mark.gpu


def lift(uv):
    return np.stack([np.sin(uv[:, 0]), np.cos(uv[:, 1]), uv[:, 0] * uv[:, 1]], 1)


def big_triangles(seed, num, extent):
    g = np.random.default_rng(seed)
    pts = g.uniform(-0.3 * extent, 1.3 * extent, (3 * num, 2))
    return pts, np.arange(3 * num, dtype=np.int32).reshape(-1, 3)


def test_raster_more_pairs_than_room(gpu, orc):
    from cvtamd import compat
    n = 400
    pts, tri = big_triangles(1, 40, n)             # most cover hundreds of the 625 tiles
    w = np.random.default_rng(2).random(len(pts))
    assert np.array_equal(compat.rasterize(pts, w, tri, 1.0, n), orc.raster(pts, w, tri, 1.0, n))


def test_locate_more_pairs_than_room(gpu):
    uv, tri = big_triangles(3, 400, 10.0)          # 15 x 15 bins, hundreds of faces per bin
    check_locate(uv, tri, np.random.default_rng(4).uniform(0, 10, (2000, 2)), lift(uv))


# the scan of the counts: one workgroup up to 16384, whole tiles of 4096 or not
@pytest.mark.parametrize("n", [16, 1009, 1024, 2032, 2048, 2064])   # 1, 4096, .. 16129, 16384, 16641 tiles
def test_raster_scan_sizes(gpu, orc, n):
    from cvtamd import compat
    uv, tri = jittered_mesh(14, n)
    uv = (uv - uv.min(0)) / (uv.max(0) - uv.min(0)).max()
    w = np.random.default_rng(n).random(len(uv))
    scale = 1.0 / max(n - 1, 1)
    assert np.array_equal(compat.rasterize(uv, w, tri, scale, n), orc.raster(uv, w, tri, scale, n))


def test_device_arguments_in_place(gpu):
    import torch
    from cvtamd import compat, recover, weighting
    uv, tri = jittered_mesh(30, 5)
    uv = uv - uv.min(0)
    p3, q = lift(uv), queries(uv, tri, 6, 1000)
    d = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (uv, p3, tri, q)]
    host_w = weighting.vertex_weights(uv, p3, tri)
    dev_w = torch.empty(len(uv), dtype=torch.float64, device="cuda")
    weighting.vertex_weights(d[0], d[1], d[2], out=dev_w)
    assert np.array_equal(dev_w.cpu().numpy(), host_w)
    host_r = compat.rasterize(uv, host_w, tri, 0.1, 300)
    dev_r = torch.empty((300, 300), dtype=torch.float32, device="cuda")
    compat.rasterize(d[0], dev_w, d[2], 0.1, 300, out=dev_r)
    assert np.array_equal(dev_r.cpu().numpy(), host_r)
    host_l = recover.locate_points(uv, tri, q, p3=p3)
    dev_l = (torch.empty(len(q), dtype=torch.int32, device="cuda"),
             torch.empty((len(q), 3), dtype=torch.float64, device="cuda"),
             torch.empty((len(q), 3), dtype=torch.float64, device="cuda"))
    recover.locate_points(d[0], d[2], d[3], p3=d[1], out=dev_l)
    for a, b in zip(dev_l, host_l):
        assert np.array_equal(a.cpu().numpy(), b)
    # the inputs were only read
    for a, b in zip(d, (uv, p3, tri, q)):
        assert np.array_equal(a.cpu().numpy(), b)


def test_outputs_over_inputs_and_unaligned(gpu):
    import torch
    from cvtamd._lib import call
    from cvtamd import recover, weighting
    uv, tri = jittered_mesh(12, 7)
    p3, q = lift(uv), queries(uv, tri, 8, 300)
    nv, nf, nq = len(uv), len(tri), len(q)
    d_uv, d_p3, d_tri = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (uv, p3, tri))
    ptr = lambda t: C.c_void_p(t.data_ptr())
    face, w, xyz = recover.locate_points(uv, tri, q, p3=p3)
    # the queries' memory receives the weights
    buf = torch.zeros(3 * nq, dtype=torch.float64, device="cuda")
    buf[:2 * nq] = torch.from_numpy(q.reshape(-1)).cuda()
    d_face = torch.empty(nq, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    call("cvt_locate_points", ptr(d_uv), None, nv, ptr(d_tri), nf, ptr(buf), nq, ptr(d_face),
         ptr(buf), None)
    assert np.array_equal(d_face.cpu().numpy(), face)
    assert np.array_equal(buf.cpu().numpy().reshape(-1, 3), w)
    # the first vertices' memory receives the vertex weights; doubles at an odd byte
    want = weighting.vertex_weights(uv, p3, tri)
    over = d_uv.clone()
    torch.cuda.synchronize()
    call("cvt_vertex_weights", ptr(over), ptr(d_p3), nv, ptr(d_tri), nf, ptr(over))
    assert np.array_equal(over.cpu().numpy().reshape(-1)[:nv], want)
    odd = torch.zeros(16 * nv + 8, dtype=torch.uint8, device="cuda")
    odd[4:4 + 16 * nv] = torch.from_numpy(np.ascontiguousarray(uv).view(np.uint8).reshape(-1)).cuda()
    got = np.empty(nv)
    torch.cuda.synchronize()
    call("cvt_vertex_weights", C.c_void_p(odd.data_ptr() + 4), ptr(d_p3), nv, ptr(d_tri), nf,
         got.ctypes.data_as(C.c_void_p))
    assert np.array_equal(got, want)


def test_bad_index_leaves_outputs(gpu):
    import torch
    from cvtamd import CvtError, compat, recover, weighting
    uv, tri = jittered_mesh(10, 9)
    bad = tri.copy()
    bad[5, 1] = len(uv)
    d_uv, d_p3, d_bad = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (uv, lift(uv), bad))
    w = torch.full((len(uv),), 7.0, dtype=torch.float64, device="cuda")
    with pytest.raises(CvtError):
        weighting.vertex_weights(d_uv, d_p3, d_bad, out=w)
    r = torch.full((64, 64), 7.0, dtype=torch.float32, device="cuda")
    with pytest.raises(CvtError):
        compat.rasterize(d_uv, w, d_bad, 0.1, 64, out=r)
    out = (torch.full((9,), 7, dtype=torch.int32, device="cuda"),
           torch.full((9, 3), 7.0, dtype=torch.float64, device="cuda"))
    with pytest.raises(CvtError):
        recover.locate_points(d_uv, d_bad, d_uv[:9], out=out)
    for t in (w, r, *out):
        assert bool((t == 7).all())


def test_threads_and_release(gpu, orc):
    from cvtamd import compat
    from cvtamd._lib import call
    jobs = []
    for k in range(6):
        uv, tri = jittered_mesh(8 + 5 * k, 20 + k)
        uv = uv - uv.min(0)
        w = np.random.default_rng(k).random(len(uv))
        jobs.append((uv, w, tri, orc.raster(uv, w, tri, 0.09, 150 + k)))
    wrong = []

    def work(k):
        uv, w, tri, want = jobs[k]
        for _ in range(5):
            if not np.array_equal(compat.rasterize(uv, w, tri, 0.09, 150 + k), want):
                wrong.append(k)
            call("cvt_release_scratch")

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
