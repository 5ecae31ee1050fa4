"""ConnectRegion on tile-local roots against the oracle where the passes turn:
one-pixel and ragged tiles, strips and tile edges crossed by one-pixel lines,
pixels outside the gray range that are regions (kept singles, also in the rows
the area count leaves out), more than 256 regions, and rows whose roots lie in
more than 64 tiles."""
import numpy as np
import pytest

import opencuda_amd as oc
import oracle

pytestmark = pytest.mark.gpu


def _check(img, min_area, max_area, roi=None):
    import torch
    t = torch.from_numpy(img).cuda()
    x1, y1, x2, y2 = roi or (0, 0, img.shape[1], img.shape[0])
    out = torch.full((y2 - y1, x2 - x1), 9, dtype=torch.uint8, device="cuda")
    oc.connect_region(oc.view(t, roi), oc.view(out), min_area, max_area)
    torch.cuda.synchronize()
    ref = oracle.connect_region(img, roi, None, min_area, max_area)
    assert np.array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("w,h", [(1, 1), (1, 300), (300, 1), (64, 64), (65, 65), (63, 129),
                                 (191, 520)])
@pytest.mark.parametrize("density", [0.3, 0.5, 0.9])
@pytest.mark.parametrize("lo,hi", [(1, 10 ** 6), (2, 40), (3, 10 ** 6)])
def test_random(device, w, h, density, lo, hi):
    rng = np.random.default_rng(w * 1000 + h + int(10 * density))
    img = np.where(rng.random((h, w)) < density, 120, 0).astype(np.uint8)
    _check(img, lo, hi)


def _spiral(n):
    img = np.zeros((n, n), np.uint8)
    x, y, dx, dy = 0, 0, 1, 0
    x0, y0, x1, y1 = 0, 0, n - 1, n - 1
    while x0 <= x1 and y0 <= y1:
        img[y, x] = 100
        nx, ny = x + dx, y + dy
        if not (x0 <= nx <= x1 and y0 <= ny <= y1):
            if dx == 1:
                y0 += 2
            elif dy == 1:
                x1 -= 2
            elif dx == -1:
                y1 -= 2
            else:
                x0 += 2
            dx, dy = -dy, dx
            nx, ny = x + dx, y + dy
            if not (0 <= nx < n and 0 <= ny < n):
                break
        x, y = nx, ny
    return img


@pytest.mark.parametrize("kind", ["spiral", "comb", "diagonals", "rings"])
def test_long_thin_regions(device, kind):
    n = 300
    yy, xx = np.mgrid[0:n, 0:n]
    img = {"spiral": lambda: _spiral(n),
           "comb": lambda: np.where((xx % 2 == 0) | (yy == n - 1), 99, 0),
           "diagonals": lambda: np.where((xx + yy) % 3 == 0, 99, 0),
           "rings": lambda: np.where(np.maximum(abs(xx - 150), abs(yy - 150)) % 2 == 0, 99, 0),
           }[kind]().astype(np.uint8)
    _check(img, 2, 10 ** 6)
    _check(img.T.copy(), 2, 10 ** 6)


@pytest.mark.parametrize("lo", [1, 2])
def test_singles_in_uncounted_rows(device, lo):
    # H = 300: the area count covers 256 rows; below it every root is kept
    rng = np.random.default_rng(3)
    img = np.where(rng.random((300, 130)) < 0.98, 60, 0).astype(np.uint8)
    _check(img, lo, 10 ** 6)


def test_many_tiles_a_row(device):
    # 70 tiles across: a row's roots and numbers run past one wave's tiles
    img = np.zeros((40, 4480), np.uint8)
    img[5:8, ::40] = 80
    img[5:8, 1::40] = 80
    img[20, 7::300] = 80
    img[21, 7::300] = 80
    _check(img, 2, 10 ** 6)


def test_pitched_roi(device):
    rng = np.random.default_rng(8)
    img = np.where(rng.random((150, 210)) < 0.6, 200, 255).astype(np.uint8)
    _check(img, 4, 10 ** 6, roi=(3, 5, 200, 149))


def test_eight_tiles_a_workgroup(device):
    # 65 x 65 tiles: past the 4,096 from which the area pass takes eight each
    rng = np.random.default_rng(17)
    img = np.full((4160, 4160), 90, np.uint8)
    img[rng.random(img.shape) < 0.02] = 0
    img[1000:1003] = 0
    img[:, 2500:2503] = 0
    img[1500:2200, 300:900] = np.where(rng.random((700, 600)) < 0.4, 90, 0)
    _check(img, 5, 10 ** 7)
