"""GPU parity of the batched full search where the bounds eliminate little and
the rest of an item is searched without them: noise under every PU shape, at
the range where that begins and at ones that do not fill the lanes, with odd
ranges, narrow MV ranges and cut windows, and where only some of an item's
bands are noise."""
import numpy as np
import pytest

from tests.test_gpu_elim import every_shape
from tests.test_gpu_elim_range import check
from tests.test_gpu_me import LAM, compare, device_cur
from xavs2_amd import lib as X
from xavs2_amd import synth

pytestmark = pytest.mark.gpu


def noise(w, h, seed):
    return np.random.default_rng(seed).integers(0, 256, (h, w)).astype(np.uint8)


@pytest.mark.parametrize("R", [23, 24, 25, 32, 43, 48, 63, 64])
def test_every_shape_on_noise(R):
    w, h = 240, 176
    check(noise(w, h, R), noise(w, h, R + 1), every_shape(w, h, R, 13, count=2), R)


@pytest.mark.parametrize("kw", [dict(mv_range_x=(-100, 131), mv_range_y=(-80, 62)), dict(mv_range_x=(9, 300)),
                                dict(mv_range_y=(-177, -20))])
@pytest.mark.parametrize("R", [27, 32])
def test_narrow_mv_ranges_on_noise(R, kw):
    w, h = 240, 176
    check(noise(w, h, 1), noise(w, h, 2), every_shape(w, h, 9, 60, count=1), R, **kw)


@pytest.mark.parametrize("spread", [300, 600])
@pytest.mark.parametrize("R", [24, 57, 62])
def test_cut_windows_on_noise(R, spread):
    w, h = 640, 512
    rng = np.random.default_rng(spread + R)
    pus = [(x, y, 16, 16) + tuple(int(v) for v in rng.integers(-spread, spread + 1, 2) // (1, 4))
           for y in range(192, 320, 32) for x in range(192, 448, 32)]
    pus += [(64, 64, 64, 64, spread, 0), (448, 192, 64, 64, 0, -spread), (64, 256, 32, 8, -spread, 40)]
    check(noise(w, h, R), noise(w, h, spread), pus, R, plain=False)


@pytest.mark.parametrize("R", [32, 64])
def test_noise_in_some_rows(R):
    """Stripes of noise in a smooth picture: bands after the first one find it."""
    w, h = 320, 256
    ref = synth.smooth_field(w, h, seed=4)
    cur = synth.multi_ref_current([ref], 16, 20, seed=5)
    for a, seed in ((ref, 6), (cur, 7)):
        n = noise(w, h, seed)
        for y in range(24, h, 80):
            a[y:y + 28] = n[y:y + 28]
    check(ref, cur, every_shape(w, h, R, 30, count=4), R)


@pytest.mark.parametrize("R", [24, 40])
def test_large_pus_of_a_large_frame(R):
    """1024 tasks and more: 16 candidate rows per lane for large PUs too."""
    w, h = 2048, 1024
    pus = [(x, y, pw, ph, 5, -9) for y in range(0, h, 64) for x in range(0, w, 64)
           for pw, ph in (((64, 64), (32, 32), (48, 64), (64, 16), (8, 32), (24, 32))[(x // 64 + y // 64) % 6],)]
    refs = []
    for r in range(2):
        d = X.DeviceRef(w, h, frac=0)
        d.load(noise(w, h, r))
        refs.append(d)
    dcur = device_cur(noise(w, h, 5))
    got = []
    for mode in (X.PLAN_BATCHED, X.PLAN_PLAIN):
        plan = X.Plan(X.me_params(w, h, R, LAM, use_fractional_me=0), X.make_pus(pus), 2, mode)
        plan.run(dcur, refs)
        got.append(plan.fetch())
    compare(got[0], got[1], pus, 2)
