"""Device memory of a triangulation context: the buffers of the points' order
exist only where points are sorted, from 65536 up."""
import pytest

pytestmark = pytest.mark.gpu


def held(max_points, contexts):
    """device memory of that many contexts"""
    import torch
    from cvtamd.delaunay import Delaunay
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    all_ = [Delaunay(max_points) for _ in range(contexts)]
    n = before - torch.cuda.mem_get_info()[0]
    for d in all_:
        d.close()
    return n


def test_no_order_buffers_below_the_order(gpu):
    held(1000, 1)                                  # the runtime's own first allocations
    # 24 bytes per point, 1.5 MB; allocations may be rounded up to 2 MB
    assert held(65536, 16) - held(65535, 16) >= 16 << 20
