"""Backwards of one scene on two streams at once, and beside a replayed graph: what each stream
enqueued is in the gradient block when its work ends (the block's copies, DevScene::rep_mask,
are folded by one stream only)."""
import numpy as np
import pytest
import torch

import scenes
from diffvg_amd import _lib

pytestmark = pytest.mark.gpu

DEV = torch.device('cuda:0')
W = H = 64


def _scene(kind):
    f = scenes.flat_case('overlap_eo')
    sc = _lib.DeviceScene(f, 0)
    if kind == 'sdf':
        d = torch.from_numpy(np.random.default_rng(3).uniform(-1, 1, (H, W, 1)).astype(np.float32)).to(DEV)
        return sc, d, lambda g, s: sc.render(W, H, 2, 2, 5, d_render_sdf=g, stream=s)
    d = torch.from_numpy(np.random.default_rng(3).uniform(-1, 1, (H, W, 4)).astype(np.float32)).to(DEV)
    return sc, d, lambda g, s: sc.render(W, H, 2, 2, 5, d_render_image=g, stream=s)


def _rel(a, b):
    return float((a - b).abs().max() / b.abs().max())


@pytest.mark.parametrize('kind', ['sdf', 'colour'])
@pytest.mark.parametrize('first', ['a', 'b'])
def test_two_streams(kind, first):
    """Stream b's adjoint is zero, so whatever it folds or adds, a's copy of the block must be
    a's gradient; then both add and the block holds twice that."""
    print('two streams', kind, first, flush=True)
    sc, d, backward = _scene(kind)
    zero = torch.zeros_like(d)
    sc.zero_grads(None)
    backward(d, None)
    want, _ = sc.grads_device(DEV, None)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    if first == 'b':
        backward(zero, b.cuda_stream)
        torch.cuda.synchronize()
    for i in range(25):
        sc.zero_grads(a.cuda_stream)
        a.synchronize()
        for _ in range(3):
            backward(zero, b.cuda_stream)
        backward(d, a.cuda_stream)
        for _ in range(3):
            backward(zero, b.cuda_stream)
        got, _ = sc.grads_device(DEV, a.cuda_stream)
        torch.cuda.synchronize()
        assert _rel(got, want) <= 1e-5, i  # float sums in another order
        sc.zero_grads(a.cuda_stream)
        a.synchronize()
        for s in (b, a):
            backward(d, s.cuda_stream)
        torch.cuda.synchronize()
        got, _ = sc.grads_device(DEV, None)
        torch.cuda.synchronize()
        assert _rel(got, 2 * want) <= 1e-5, i


def test_beside_a_replayed_graph():
    print('two streams, graph', flush=True)
    sc, d, backward = _scene('sdf')
    zero = torch.zeros_like(d)
    sc.zero_grads(None)
    backward(d, None)
    want, _ = sc.grads_device(DEV, None)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    block = torch.empty_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=a):
        backward(d, a.cuda_stream)
    for i in range(10):
        sc.zero_grads(None)
        torch.cuda.synchronize()
        backward(zero, b.cuda_stream)
        with torch.cuda.stream(a):
            g.replay()
        for _ in range(3):
            backward(zero, b.cuda_stream)
        with torch.cuda.stream(a):
            got, _ = sc.grads_device(DEV, a.cuda_stream)
            block.copy_(got)
        torch.cuda.synchronize()
        assert _rel(block, want) <= 1e-5, i
