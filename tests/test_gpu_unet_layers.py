"""GPU checks of the warm-start network's convolutions at the edges of their
tiles: images narrower than a strip, sides that are no multiple of the tile
at any level, and enough images for every tile shape and pixel split."""
import numpy as np
import pytest

from test_gpu_unet import setup_net

pytestmark = pytest.mark.gpu


def nontrivial_head(net, p, ref, seed):
    who = ref.layout(len(p))[2]
    p[who:who + 2 * ref.HEAD_C] = np.random.default_rng(seed).normal(0, 0.2, 2 * ref.HEAD_C)
    net.set_params(p.astype(np.float32))
    return p.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("R,N", [(8, 1), (8, 5), (40, 1), (40, 13), (72, 26)])
def test_forward_at_tile_edges(gpu, R, N):
    from oracle import unet_ref as ref
    net, p, x = setup_net(R, N, 21)
    p = nontrivial_head(net, p, ref, 22)
    net.forward(N)
    f = net.field(N)
    fr, _ = ref.forward(p, x, rb=True)
    assert np.abs(f - fr).max() < 2e-2 * np.abs(fr).max()


@pytest.mark.parametrize("R,N", [(8, 1), (40, 1), (40, 11), (72, 4)])
def test_gradients_at_tile_edges(gpu, R, N):
    from oracle import unet_ref as ref
    S = 2 * R
    net, p, x = setup_net(R, N, 23)
    p = nontrivial_head(net, p, ref, 24)
    g = np.random.default_rng(25)
    uv = g.random((N, S, 2)).astype(np.float32)
    tgt = g.normal(0, 0.05, (N, S, 2)).astype(np.float32)
    net.forward(N)
    net.loss_backward(N, uv, tgt, S)
    grad = net.grads().astype(np.float64)
    fr, cache = ref.forward(p, x, rb=True)
    _, gf = ref.loss_and_grad_field(fr, uv.astype(np.float64), tgt.astype(np.float64))
    gr = ref.backward(p, cache, gf, rb=True)
    assert np.linalg.norm(grad - gr) < 0.1 * np.linalg.norm(gr)
    wo, bo = ref.layout(len(p))[:2]
    ends = wo[1:] + [ref.layout(len(p))[2]]
    for l in range(14):
        for a, b in ((wo[l], bo[l]), (bo[l], ends[l])):   # weights, biases
            u, v = grad[a:b], gr[a:b]
            assert u @ v > 0.98 * np.linalg.norm(u) * np.linalg.norm(v), l
