"""The unrolled kernels at every radius they serve, against the oracle and
against the run-time tap list (the same taps with a template the library does
not recognise as the canonical one: a weight past the radius changed).  Halo
classes end at 4, 8, 12, 16 and 20; from r = 16 the weight table no longer
fits in LDS as a whole."""
import numpy as np
import pytest

import opencuda_amd as oc
import oracle
from opencuda_amd import surrogate as sg
from tests._gpu import check_against_oracle, run_exact

pytestmark = pytest.mark.gpu

RADII = [1, 2, 4, 5, 8, 9, 10, 12, 13, 14, 16, 17, 18, 19, 20]


def _img(w, h, seed):
    return oc.synth_image(w, h, 14, 6, 70, 12.0, seed)


def _luts(ss, sr):
    off, w = oc.gauss_template(ss)
    rng = oc.euclid_template(sr)
    other = w.copy()
    other[-1] += 1.0                      # past every radius the tests use
    return oc.Lut(off, w, rng), oc.Lut(off, other, rng)


@pytest.mark.parametrize("mode", [oc.MODE_REF, oc.MODE_STD])
@pytest.mark.parametrize("r", RADII)
def test_single_image(device, r, mode):
    if mode == oc.MODE_REF and r == 20:
        pytest.skip("REF reads past the template at r = 20")
    img = _img(203, 139, r)
    ss, sr = max(0.6, r / 1.5), 20.0 + r
    ring, taps = _luts(ss, sr)
    got = run_exact(img, r, ss, sr, mode, lut=ring)
    check_against_oracle(img, r, ss, sr, mode, got=got)
    if r < 20:
        assert np.array_equal(got, run_exact(img, r, ss, sr, mode, lut=taps))


@pytest.mark.parametrize("config", [0, 1])
@pytest.mark.parametrize("top", [4, 8, 12, 16])
def test_batch_of_all_radii_of_a_halo(device, top, config):
    import torch
    imgs, outs, luts, jobs, want = [], [], [], [], []
    for r in range(max(1, top - 5), top + 1):
        for mode in (oc.MODE_REF, oc.MODE_STD):
            img = _img(90 + 7 * r, 70 + 3 * r, 100 + r)
            ss, sr = max(0.6, r / 1.5), 20.0 + r
            imgs.append(torch.from_numpy(img).cuda())
            outs.append(torch.zeros_like(imgs[-1]))
            luts.append(oc.Lut.from_sigmas(ss, sr))
            jobs.append(oc.Job(oc.view(imgs[-1]), oc.view(outs[-1]), luts[-1].handle, r, mode))
            want.append(oracle.filter(img, r, ss, sr, mode=mode))
    b = oc.Batch(jobs, config)
    assert b.unrolled
    b.run()
    torch.cuda.synchronize()
    for o, w in zip(outs, want):
        assert np.array_equal(o.cpu().numpy(), w)


@pytest.mark.parametrize("mode", [oc.MODE_REF, oc.MODE_STD])
@pytest.mark.parametrize("r", [8, 9, 12, 13, 16, 17])
def test_surrogate_check_and_fallback(device, r, mode):
    import torch
    net = sg.Surrogate(seed=1)
    net.load(sg.DEFAULT_WEIGHTS)
    img = torch.from_numpy(_img(330, 270, 7)).cuda()
    res = []
    for lut in _luts(r / 1.5, 30.0):
        out = torch.zeros_like(img)
        counts = net.filter(oc.view(img), oc.view(out), lut, r, mode, 30.0, 2)
        torch.cuda.synchronize()
        res.append((counts, out.cpu().numpy()))
    assert res[0][0] == res[1][0]
    assert np.array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("mode", [oc.MODE_REF, oc.MODE_STD])
@pytest.mark.parametrize("r,w,h", [(10, 1100, 1000), (13, 1100, 1000), (16, 1100, 1000),
                                   (17, 1100, 1000), (18, 1100, 1000),
                                   (3, 1021, 767), (4, 1100, 1000), (7, 1021, 767), (8, 1700, 1300)])
def test_images_past_the_small_tiles(device, r, w, h, mode):
    # Images of several rounds of tiles.  Which kernel an image takes, and every
    # kernel at sizes that take it: test_gpu_exact_plan.py.  (REF r = 17 and 18
    # take the tap list themselves here.)
    ring, taps = _luts(r / 1.5, 30.0)
    img = _img(w, h, r)
    got = run_exact(img, r, 0, 0, mode, lut=ring)
    assert np.array_equal(got, run_exact(img, r, 0, 0, mode, lut=taps))
