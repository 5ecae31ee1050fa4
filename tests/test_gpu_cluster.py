"""LocalCluster's two-phase kernel against the oracle where its branches turn:
pixels settled by the first step or queued, every tile height, rows read as
dwords or clamped byte by byte, misaligned pitches, kept counts from 1 to 8
and the counts outside that range."""
import numpy as np
import pytest

import opencuda_amd as oc
import oracle

pytestmark = pytest.mark.gpu


def _run(img, roi, whole_alloc, rng, cnt, gap, diffe):
    import torch
    t = torch.from_numpy(img).cuda()
    x1, y1, x2, y2 = roi
    out = torch.full((y2 - y1, x2 - x1), 3, dtype=torch.uint8, device="cuda")
    alloc = oc.alloc_range(t, roi) if whole_alloc else (0, 0)
    oc.local_cluster(oc.view(t, roi), oc.view(out), rng, cnt, gap, diffe, alloc=alloc)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _content(kind, h, w):
    if kind == "flat":
        return np.full((h, w), 90, np.uint8)
    noise = {"quiet": 1.5, "noisy": 10.0}[kind]
    return oc.synth_image(w, h, max(4, w * h // 6000), 4, 64, noise, 31 + h)


@pytest.mark.parametrize("kind", ["flat", "quiet", "noisy"])
@pytest.mark.parametrize("w,h,pad", [(63, 17, 1), (65, 33, 2), (131, 66, 3), (260, 128, 0)])
@pytest.mark.parametrize("rng,cnt", [(2, 1), (8, 5), (8, 8), (16, 7), (1, 5)])
def test_small_tiles(device, kind, w, h, pad, rng, cnt):
    img = _content(kind, h + 4, w + 4 + pad)
    roi = (3, 2, 3 + w, 2 + h)
    got = _run(img, roi, True, rng, cnt, 10, 10)
    assert np.array_equal(got, oracle.local_cluster(img, roi, pntrange=rng, pntcount=cnt))


@pytest.mark.parametrize("h", [1100, 2113])        # 32-row and 64-row tiles on 256 CUs
def test_tall_tiles(device, h):
    img = _content("noisy", h, 2051)
    got = _run(img, (0, 0, 2051, h), False, 8, 5, 10, 10)
    assert np.array_equal(got, oracle.local_cluster(img, pntrange=8, pntcount=5))


@pytest.mark.parametrize("cnt", [9, 12])           # more averages kept than there are
def test_counts_beyond_the_directions(device, cnt):
    img = _content("quiet", 70, 90)
    got = _run(img, (0, 0, 90, 70), True, 8, cnt, 10, 10)
    assert np.array_equal(got, oracle.local_cluster(img, pntrange=8, pntcount=cnt))
