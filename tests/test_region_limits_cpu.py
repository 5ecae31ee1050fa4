"""ConnectRegion refuses, before any GPU work, the images its launches cannot
cover: 2^26 rows and more (64 threads a row reach the 2^32 threads a launch
may hold) and more pixels than a 32-bit label numbers.  The views' addresses
are never read."""
import pytest

import opencuda_amd as oc


@pytest.mark.parametrize("w,h", [(1, 1 << 26), (31, 1 << 26), (2, (1 << 30) - 1), (1, 2 ** 31 - 1)])
def test_too_tall(w, h):
    v, o = oc.View(1 << 20, w, h, w), oc.View(1 << 40, w, h, w)
    with pytest.raises(oc.BfError) as e:
        oc.connect_region(v, o, 1, 100, stream=0)
    assert e.value.code == oc.INVALID_DATA and "rows" in str(e.value)


def test_too_many_pixels():
    v, o = oc.View(1 << 20, 65536, 32768, 65536), oc.View(1 << 40, 65536, 32768, 65536)
    with pytest.raises(oc.BfError) as e:
        oc.connect_region(v, o, 1, 100, stream=0)
    assert e.value.code == oc.INVALID_DATA and "labels" in str(e.value)
