"""The tile pass of ConnectRegion (csrc/region.hip) restated on Python
integers, against scipy's 8-connected labels: a run hooks onto the first run
above that it touches, pointer jumping (seven rounds, then walks), unions of the
runs that touch a second run above; the shortcut for tiles of at most one run a
row; the masks' bit rules; the areas' paired 16-bit counters."""
import numpy as np
import pytest
from scipy import ndimage

M64 = (1 << 64) - 1
ROWS = 64


def starts(m):
    return m & ~(m << 1) & M64


def run_bits(m, s):
    return m & ~(m + s) & ~(s - 1) & M64


def touched(m, u, s):
    r = run_bits(m, s)
    return u & (r | (r << 1) | (r >> 1)) & M64


def run_of(m, t):
    return bin(starts(m) & (t ^ (t - 1))).count("1") - 1


def bits(m):
    while m:
        b = m & -m
        yield b
        m ^= b


def masks_of(tile):
    return [sum(1 << int(x) for x in np.flatnonzero(row)) for row in tile]


def tile_pass(masks):
    """{(row, run): root (row, run)} and areas by root."""
    parent, extra = {}, []
    for y, m in enumerate(masks):
        u = masks[y - 1] if y else 0
        for k, s in enumerate(bits(starts(m))):
            t = touched(m, u, s)
            parent[y, k] = (y - 1, run_of(u, t)) if t else (y, k)
            more = starts(u) & t & (t - 1)              # runs past the first touched column
            extra += [((y, k), (y - 1, run_of(u, b))) for b in bits(more)]
    for _ in range(7):
        parent = {r: parent[p] for r, p in parent.items()}

    def unite(a, b):
        while a != b:
            pa, pb = parent[a], parent[b]
            if (pa, pb) != (a, b):
                a, b = pa, pb
            else:
                parent[max(a, b)] = min(a, b)
                return

    for a, b in extra:
        unite(parent[a], b)
    root = {}
    for r in parent:
        p = r
        while parent[p] != p:
            p = parent[p]
        root[r] = p
    return root


def one_run_rows(masks):
    """The shortcut: a row's component starts at the last row at or above it
    that touches nothing above."""
    breaks = [y for y, m in enumerate(masks)
              if not ((masks[y - 1] if y else 0) & (m | (m << 1) | (m >> 1)) & M64)]
    return {(y, 0): (max(b for b in breaks if b <= y), 0) for y, m in enumerate(masks) if m}


def check(tile):
    masks = masks_of(tile)
    label, n = ndimage.label(tile, structure=np.ones((3, 3)))
    root = tile_pass(masks)
    if all(starts(m) & (starts(m) - 1) == 0 for m in masks):
        assert one_run_rows(masks) == root
    # two 16-bit areas a 32-bit word, as the kernel's table of 33 run entries a row
    cnt = [0] * (ROWS * 33 // 2)
    first = {}
    for (y, k), p in root.items():
        s = list(bits(starts(masks[y])))[k]
        run = run_bits(masks[y], s)
        x = s.bit_length() - 1
        assert run == sum(1 << c for c in range(x, x + bin(run).count("1")))
        first.setdefault(p, label[y, x])
        assert label[y, x] == first[p]                  # one label a root
        at = p[0] * 33 + p[1]
        cnt[at >> 1] += bin(run).count("1") << (16 * (at & 1))
        assert cnt[at >> 1] <= 0xFFFFFFFF
        for c in np.flatnonzero(tile[y]):
            if (run >> int(c)) & 1:
                assert run_of(masks[y], 1 << int(c)) == k
    assert len(set(first.values())) == len(first) == n  # and one root a label
    for p, lab in first.items():
        at = p[0] * 33 + p[1]
        assert (cnt[at >> 1] >> (16 * (at & 1))) & 0xFFFF == (label == lab).sum()
        ys, xs = np.nonzero(label == lab)               # the root is the first pixel's run
        assert p[0] == ys[0] and run_of(masks[ys[0]], 1 << int(xs[0])) == p[1]


@pytest.mark.parametrize("density", [0.05, 0.2, 0.4, 0.5, 0.6, 0.8, 0.97, 1.0])
@pytest.mark.parametrize("seed", range(3))
def test_random_tiles(density, seed):
    check(np.random.default_rng(100 * seed + int(100 * density)).random((ROWS, 64)) < density)


@pytest.mark.parametrize("kind", ["comb", "comb_up", "diagonal", "anti", "checker", "rings", "zigzag", "empty"])
def test_shapes(kind):
    y, x = np.mgrid[0:ROWS, 0:64]
    check({"comb": (x % 2 == 0) | (y == 63), "comb_up": (x % 2 == 0) | (y == 0), "diagonal": x == y,
           "anti": x == 63 - y, "checker": (x + y) % 2 == 0, "rings": np.maximum(abs(x - 32), abs(y - 31)) % 2 == 0,
           "zigzag": x == abs((y % 20) - 10) + 5, "empty": x < 0}[kind])


@pytest.mark.parametrize("seed", range(20))
def test_one_run_a_row(seed):
    rng = np.random.default_rng(seed)
    tile = np.zeros((ROWS, 64), bool)
    a, n = 20, 10
    for y in range(ROWS):
        a = int(np.clip(a + rng.integers(-6, 7), 0, 63))
        n = int(rng.integers(0 if rng.random() < 0.1 else 1, 12))
        tile[y, a:a + n] = True
    check(tile)
