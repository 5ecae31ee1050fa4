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


def test_costs_of_the_kernel_that_runs(device, tuned):
    # a batch on the canonical template, a batch on another one, one image of it
    unrolled, taps, batch_taps = [5.0] * 9, [5.0] * 9, [5.0] * 9
    unrolled[0], taps[5], batch_taps[4] = 1.0, 2.0, 2.0
    for r, mode in ((10, STD), (4, REF)):
        tuned.install(r, mode, unrolled, taps, batch_taps)
        assert tuned.get(r, mode) == (0, unrolled)
        assert tuned.get_taps(r, mode) == (5, taps, batch_taps)
        b = _Batch([(r, mode)])
        assert b.batch.unrolled and b.batch.config == 0
        b.check()
        b = _Batch([(r, mode)], custom=True)
        assert not b.batch.unrolled and b.batch.config == 4
        b.check()
        assert oc.exact_plan(b.keep[0][2], r, mode, 8192, 8192) == (5, False)
    mixed = _Batch([(10, STD), (4, REF)], custom=True)
    assert mixed.batch.config == 4
    mixed.check()


def test_measured_costs(device, tuned):
    best, cost = tuned.tune(5, STD, 512, 256, reps=1)
    tbest, taps, batch_taps = tuned.get_taps(5, STD)
    assert cost[best] == min(cost) > 0 and taps[tbest] == min(taps) > 0
    assert batch_taps[2:] == cost[2:]        # the unrolled kernels have configurations 0 and 1
    assert cost[0] != batch_taps[0] and cost[1] != batch_taps[1]


def test_a_table_of_one_cost_serves_all_launches(device, tuned):
    cost = [3.0] * 9
    cost[6] = 1.0
    tuned.install(7, STD, cost)
    assert tuned.get(7, STD) == (6, cost) and tuned.get_taps(7, STD) == (6, cost, cost)


def test_custom_template_takes_the_measured_configuration(device, tuned):
    # r = 16: no more rows than the canonical table the cost was measured with
    cost = [2.0] * 9
    cost[4] = 1.0
    tuned.install(16, STD, cost)
    b = _Batch([(16, STD)], custom=True)
    assert not b.batch.unrolled and b.batch.config == 4
    b.check()
    assert oc.exact_plan(b.keep[0][2], 16, STD, 8192, 8192) == (4, False)


def test_tuned_costs_on_an_image_of_few_tiles(device, tuned):
    # 1021 x 767 on 256 CUs: two 128 x 16 tiles or three 64 x 16 ones a CU, so
    # 64 x 16 tiles are taken where they cost less than 1.2 of the others; the
    # default (64 x 32 here) stands where it costs at most 3% more than the best
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are chosen for 256 CUs")
    lut = _Batch([(6, STD)], custom=True).keep[0][2]
    for costs, small, large in (({3: 1.15, 4: 1.0}, 3, 4), ({3: 1.25, 4: 1.0}, 4, 4), ({1: 1.02, 4: 1.0}, 1, 1),
                                ({1: 1.05, 4: 1.0}, 4, 4)):
        cost = [9.0] * 9
        for c, k in costs.items():
            cost[c] = k
        tuned.install(6, STD, cost)
        assert oc.exact_plan(lut, 6, STD, 1021, 767) == (small, False)
        assert oc.exact_plan(lut, 6, STD, 4096, 4096) == (large, False)


def test_default_stands_within_two_percent(device, tuned):
    for default, config in ((1.015, 0), (1.03, 1)):
        for r, mode in ((15, STD), (7, STD)):
            cost = [9.0] * 9
            cost[0], cost[1] = default, 1.0
            tuned.install(r, mode, cost)
        b = _Batch([(15, STD), (7, STD)])
        assert b.batch.config == config and b.batch.unrolled
        b.check()
