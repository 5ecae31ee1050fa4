"""In-place filtering for odd and even pass counts (an even count starts in
the image itself, an odd one in a copy), with and without caller scratch, on a
ROI of a pitched image whose other pixels stay as they are."""
import numpy as np
import pytest

import opencuda_amd as oc
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scratch", [False, True])
@pytest.mark.parametrize("repeat", [1, 2, 3, 4])
def test_passes(device, repeat, scratch):
    import torch
    img = oc.synth_image(157, 98, 12, 4, 40, 12.0, 5)
    x1, y1, x2, y2 = 5, 3, 150, 95
    t = torch.from_numpy(img).cuda()
    work = torch.empty((x2 - x1) * (y2 - y1), dtype=torch.uint8, device="cuda") if scratch else None
    lut = oc.Lut.from_sigmas(2.5, 25.0)
    oc.exact_inplace(oc.view(t, (x1, y1, x2, y2)), lut, 4, oc.MODE_STD, repeat, work=work)
    torch.cuda.synchronize()
    want = img.copy()
    sub = want[y1:y2, x1:x2].copy()
    for _ in range(repeat):
        sub = oracle.filter(sub, 4, 2.5, 25.0, mode=oracle.STD)
    want[y1:y2, x1:x2] = sub
    assert np.array_equal(t.cpu().numpy(), want)
