"""Weight gradients where a workgroup walks many rows of a strip (the rings of
rows in LDS wrap, runs have odd lengths and cross strips and crops), per layer
and per W / b.

* Against the float64 network with the GPU's BF16 rounding points.  What the
  reference leaves out is the rounding of the gradients passed down, at most
  2^-9 of an element (1.1e-3 rms) in each of five layers: 2.5e-3 of a tensor's
  norm where its sums cancel (targets are noise, so they do), so 1% at four
  times that.  One lost row of 255 changes a cancelling sum by 6%.
* Against itself: the gradients of 8 crops are the mean of those of each crop
  alone, whose rows are about as many as the workgroups.  Crops of a power of
  two scale exactly, so only the order of FP32 sums differs: for K = 8 x 255 x
  130 terms 0.2 sqrt(K) 2^-24 = 6e-6 of the norm in one chain, less in the
  kernel's; 1e-4 here.  One lost pixel is 1 / sqrt(K) = 2e-3."""
import numpy as np
import pytest

from opencuda_amd import surrogate as sg
from tests.test_gpu_surrogate import LAYERS, _reference

pytestmark = pytest.mark.gpu


def _inputs(n, h, w):
    rng = np.random.default_rng(n * 10000 + h * 10 + w)
    x = rng.integers(0, 256, (n, h, w)).astype(np.uint8)
    y = rng.integers(0, 256, (n, h, w)).astype(np.uint8)
    return x, y, (rng.random(n) * 30 + 15).astype(np.float32)


def _net():
    net = sg.Surrogate(seed=3)
    p = net.get_params()
    net.set_params(p + np.random.default_rng(1).normal(0, 0.02, p.size).astype(np.float32))
    return net


def _grads(net, x, y, sigma):
    import torch
    _, g, _ = net.forward_backward(*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, y, sigma)))
    torch.cuda.synchronize()
    return g.cpu().double().numpy()


def _each_tensor(got, ref, tol):
    o = 0
    for layer, (cin, cout) in enumerate(LAYERS):
        for name, size in (("W", 9 * cin * cout), ("b", cout)):
            a, b = got[o:o + size], ref[o:o + size]
            o += size
            err = np.linalg.norm(a - b) / np.linalg.norm(b)
            assert err < tol, f"layer {layer} {name}: {err:.2e}"
    assert o == got.size


@pytest.mark.parametrize("n,h,w", [(6, 255, 130), (4, 301, 70), (1, 2051, 64), (3, 600, 63)])
def test_against_float64(device, n, h, w):
    x, y, sigma = _inputs(n, h, w)
    net = _net()
    _, ref, _ = _reference(net.get_params(), x, y, sigma)
    _each_tensor(_grads(net, x, y, sigma), ref, 1e-2)


@pytest.mark.parametrize("h,w", [(255, 130), (256, 256), (77, 200), (767, 61), (30, 513)])
def test_crops_together_and_alone(device, h, w):
    x, y, sigma = _inputs(8, h, w)
    net = _net()
    alone = sum(_grads(net, x[i:i + 1], y[i:i + 1], sigma[i:i + 1]) for i in range(8)) / 8
    _each_tensor(_grads(net, x, y, sigma), alone, 1e-4)
