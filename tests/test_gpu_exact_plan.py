"""Every unrolled single-image kernel at sizes that bf_exact gives to it (the
plan is asserted, on the 256 CUs its rule counts in), against the tap-list
kernel on the same image: same bits.  The kernels are named by tile (config 3
64 x 16, 1 64 x 32, 0 64 x 64) and staged halo (4 to r = 4, 8 to 8, ...)."""
import numpy as np
import pytest

import opencuda_amd as oc

pytestmark = pytest.mark.gpu

REF, STD = oc.MODE_REF, oc.MODE_STD
CUS = 256


def _both(w, h, r, mode, config, unrolled=True):
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != CUS:
        pytest.skip("the sizes are chosen for 256 CUs")
    lut = oc.Lut.from_sigmas(max(0.6, r / 1.5), 20.0 + r)
    assert oc.exact_plan(lut, r, mode, w, h) == (config, unrolled)
    g = torch.Generator(device="cuda").manual_seed(1000 * r + w)
    base = torch.linspace(20, 220, w, device="cuda").expand(h, w)
    img = (base + 12.0 * torch.randn((h, w), generator=g, device="cuda")).round().clamp(0, 255).to(torch.uint8)
    got, want = torch.full_like(img, 3), torch.full_like(img, 5)
    oc.exact(oc.view(img), oc.view(got), lut, r, mode)
    oc.exact(oc.view(img), oc.view(want), lut, r, mode, config=2 if r < 16 else 3)
    torch.cuda.synchronize()
    bad = int((got != want).sum())
    assert bad == 0, f"{bad} of {w * h} pixels differ"


@pytest.mark.parametrize("mode", [REF, STD])
@pytest.mark.parametrize("r,w,h", [(1, 203, 139), (4, 1021, 767), (4, 65, 17), (5, 203, 139),
                                   (6, 800, 801), (7, 1021, 767), (8, 511, 509)])
def test_64x16(device, r, w, h, mode):
    _both(w, h, r, mode, 3)


@pytest.mark.parametrize("mode", [REF, STD])
@pytest.mark.parametrize("r,w,h", [(1, 2047, 1535), (2, 2048, 1536), (3, 2047, 2049), (4, 2047, 1535),
                                   (5, 1601, 1203), (6, 1601, 1203), (7, 2048, 2047), (8, 2047, 1535),
                                   (9, 203, 139), (9, 1700, 1301), (10, 501, 499), (12, 1101, 1099),
                                   (13, 700, 701), (16, 701, 700)])
def test_64x32(device, r, w, h, mode):
    _both(w, h, r, mode, 1)


@pytest.mark.parametrize("r,w,h", [(17, 203, 139), (18, 701, 699), (19, 1101, 1099), (20, 500, 500)])
def test_64x32_largest_radii(device, r, w, h):
    _both(w, h, r, STD, 1)


@pytest.mark.parametrize("mode", [REF, STD])
@pytest.mark.parametrize("r,w,h", [(10, 1000, 1001), (11, 999, 1000), (12, 1301, 1299), (13, 1000, 1001),
                                   (14, 1300, 1301), (16, 1001, 999)])
def test_64x64(device, r, w, h, mode):
    _both(w, h, r, mode, 0)


@pytest.mark.parametrize("r,w,h", [(17, 1000, 1001), (18, 1301, 1299), (19, 1001, 999), (20, 1300, 1301)])
def test_64x64_largest_radii_std(device, r, w, h):
    _both(w, h, r, STD, 0)


@pytest.mark.parametrize("r", [17, 18, 19])
def test_64x64_largest_radii_ref(device, r):
    _both(4097, 4095, r, REF, 0)


@pytest.mark.parametrize("r", [17, 18, 19])
def test_tap_list_below(device, r):
    _both(1101, 1099, r, REF, 3, unrolled=False)


@pytest.mark.parametrize("mode", [REF, STD])
@pytest.mark.parametrize("w,h,config", [(512, 512, 3), (1024, 256, 3), (513, 512, 1), (800, 800, 1),
                                        (1021, 767, 1), (1700, 1300, 1)])
def test_r8_tiles(device, w, h, config, mode):
    # two 64 x 16 workgroups fit a CU: only images of one tile a CU take them
    _both(w, h, 8, mode, config)


@pytest.mark.parametrize("w,h,config", [(1021, 767, 3), (1279, 1024, 3), (1500, 1150, 1), (1700, 1300, 1),
                                        (1900, 1400, 1)])
def test_r7_ref_tiles(device, w, h, config):
    # from seven 64 x 16 tiles a CU on, quiet images lose on them
    _both(w, h, 7, REF, config)


@pytest.mark.parametrize("r,mode,config", [(12, STD, 1), (13, STD, 0), (15, STD, 0), (16, STD, 0), (18, STD, 1),
                                           (12, REF, 1), (13, REF, 1), (15, REF, 1), (16, REF, 1)])
def test_three_rounds_against_two(device, r, mode, config):
    # 1100 x 1100: three rounds of 64 x 32 tiles or two of 64 x 64
    _both(1100, 1100, r, mode, config)


@pytest.mark.parametrize("r", [5, 6])
@pytest.mark.parametrize("w,h,mode,config", [(1021, 767, REF, 3), (1279, 1024, REF, 1), (1700, 1300, REF, 1),
                                             (1279, 1024, STD, 3), (1700, 1300, STD, 3), (1600, 1200, STD, 1)])
def test_r5_r6_tiles(device, r, w, h, mode, config):
    _both(w, h, r, mode, config)


@pytest.mark.parametrize("r", [17, 19])
@pytest.mark.parametrize("w,h,unrolled", [(3001, 2999, False), (3300, 3300, True)])
def test_ref_largest_radii_by_size(device, r, w, h, unrolled):
    _both(w, h, r, REF, 0 if unrolled else 3, unrolled)


def test_plan_refuses(device):
    lut = oc.Lut.from_sigmas(2.0, 20.0)
    for r, mode, w, h in ((0, REF, 9, 9), (21, STD, 9, 9), (20, REF, 9, 9), (3, 2, 9, 9), (3, REF, 0, 9)):
        with pytest.raises(oc.BfError) as e:
            oc.exact_plan(lut, r, mode, w, h)
        assert e.value.code == oc.INVALID_DATA
