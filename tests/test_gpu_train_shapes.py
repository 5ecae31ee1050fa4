"""Weight gradients over crops whose rows and strips split unevenly over the
workgroups: strips of 1 to 64 columns, fewer rows than workgroups, runs that
cross columns and crops, against autograd in float64 with BF16 rounding points
left out (so within the BF16 error that the full-size check allows)."""
import numpy as np
import pytest

from opencuda_amd import surrogate as sg

pytestmark = pytest.mark.gpu


def _layers(p):
    out, at = [], 0
    for layer in range(6):
        cin, cout = (2 if layer == 0 else 32), (1 if layer == 5 else 32)
        out.append((p[at:at + 9 * cin * cout].reshape(9, cin, cout),
                    p[at + 9 * cin * cout:at + 9 * cin * cout + cout]))
        at += 9 * cin * cout + cout
    return out


@pytest.mark.parametrize("n,h,w", [(1, 13, 13), (1, 14, 64), (2, 33, 65), (5, 70, 129), (3, 200, 77)])
def test_gradients(device, n, h, w):
    import torch
    g = torch.Generator().manual_seed(n * 1000 + h)
    x = torch.randint(0, 256, (n, h, w), dtype=torch.uint8, generator=g)
    y = torch.randint(0, 256, (n, h, w), dtype=torch.uint8, generator=g)
    sigma = torch.rand(n, generator=g) * 30 + 15
    net = sg.Surrogate(seed=3)
    _, grads, _ = net.forward_backward(x.cuda(), y.cuda(), sigma.cuda())
    p = torch.from_numpy(net.get_params().astype(np.float64)).requires_grad_(True)
    u = x.double() / 255.0
    a = torch.stack([u, (sigma.double() / 100.0)[:, None, None].expand_as(u)], -1)
    for k, (wt, b) in enumerate(_layers(p)):
        q = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        acc = b
        for t in range(9):
            acc = acc + q[:, t // 3:t // 3 + h, t % 3:t % 3 + w] @ wt[t]
        a = acc.relu() if k < 5 else acc
    d = (u + a[..., 0] - y.double() / 255.0)[:, 6:h - 6, 6:w - 6]
    ((d * d).sum() / d.numel()).backward()
    ref, got = p.grad.numpy(), grads.cpu().double().numpy()
    # BF16 operands: 2^-9 relative a factor, some tens of roundings in a chain
    # of six layers and back
    assert np.linalg.norm(got - ref) < 0.06 * np.linalg.norm(ref)
