"""The configuration and kernels that a batch takes by itself (config < 0):
tables that do not fit in LDS whole (from r = 16) keep neither the unrolled
kernels nor a measured configuration from it."""
import numpy as np
import pytest

import opencuda_amd as oc
import oracle
from opencuda_amd import autotune

pytestmark = pytest.mark.gpu

REF, STD = oc.MODE_REF, oc.MODE_STD


class _Batch:
    """A batch of one image a (radius, mode) pair; custom: on a template that
    is not the canonical one (a weight past every radius changed)."""

    def __init__(self, pairs, config=-1, custom=False, size=(210, 150)):
        import torch
        self.want, self.keep, jobs = [], [], []
        for r, mode in pairs:
            img = oc.synth_image(size[0], size[1], 14, 6, 70, 12.0, 100 + r)
            ss, sr = max(0.6, r / 1.5), 20.0 + r
            off, w = oc.gauss_template(ss)
            if custom:
                w[-1] += 1.0
            lut = oc.Lut(off, w, oc.euclid_template(sr))
            tin = torch.from_numpy(img).cuda()
            out = torch.zeros_like(tin)
            self.keep.append((tin, out, lut))
            jobs.append(oc.Job(oc.view(tin), oc.view(out), lut.handle, r, mode))
            self.want.append(oracle.filter(img, r, ss, sr, mode=mode))
        self.batch = oc.Batch(jobs, config)

    def check(self):
        import torch
        self.batch.run()
        torch.cuda.synchronize()
        for (_, out, _), w in zip(self.keep, self.want):
            assert np.array_equal(out.cpu().numpy(), w)


@pytest.fixture
def tuned():
    autotune.reset()
    yield autotune
    autotune.reset()


@pytest.mark.parametrize("pairs", [[(16, REF)], [(16, STD)], [(3, STD), (9, REF), (16, STD)],
                                   [(r, m) for r in range(11, 17) for m in (REF, STD)]])
def test_r16_by_default(device, tuned, pairs):
    b = _Batch(pairs)
    assert b.batch.unrolled and b.batch.config == 0
    b.check()


@pytest.mark.parametrize("config", range(9))
@pytest.mark.parametrize("mode", [REF, STD])
def test_r16_takes_the_measured_configuration(device, tuned, mode, config):
    cost = [2.0] * 9
    cost[config] = 1.0
    tuned.install(16, mode, cost)
    b = _Batch([(16, mode)])
    assert b.batch.config == config
    assert b.batch.unrolled == (config == 0 or (config == 1 and mode == STD))
    b.check()


def test_custom_template_keeps_a_configuration_its_table_fits(device, tuned):
    b = _Batch([(16, STD)], custom=True)
    assert not b.batch.unrolled and b.batch.config == 2
    b.check()


@pytest.mark.parametrize("pairs,unrolled", [([(16, REF)], False), ([(16, STD)], True), ([(15, REF)], True),
                                            ([(16, REF), (16, STD)], False),
                                            ([(16, REF), (15, REF), (16, STD)], False),
                                            ([(16, REF), (15, REF), (16, STD), (14, STD)], True)])
def test_ref_r16_on_64x32_tiles(device, pairs, unrolled):
    # the tap list where REF r = 16 is more than a third of the pixel-taps
    b = _Batch(pairs, config=1)
    assert b.batch.unrolled == unrolled
    b.check()
