"""GPU parity of the batched full search (successive elimination up to R = 64)
with the oracle and with the plain plan's exhaustive search, where it can go
wrong: every PU shape at ranges around the kernel's splits (4 and 16 candidate
rows per lane, columns that do not fill a lane pair or a row group, one or
several bands), search centres of both parities, pictures on which no candidate
is eliminated, on which all tie, or on which one matches exactly, narrow MV
ranges, and windows that are cut or do not fit the LDS with their sums."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_me import LAM, compare, device_cur, oracle_ref, oracle_results
from xavs2_amd import lib as X
from xavs2_amd import synth

pytestmark = pytest.mark.gpu


def pictures(kind, w, h, seed):
    rng = np.random.default_rng(seed)
    if kind == "noise":      # bounds far below the SADs: every tile is costed
        return rng.integers(0, 256, (h, w)).astype(np.uint8), rng.integers(0, 256, (h, w)).astype(np.uint8)
    if kind == "flat":       # costs differ by their rates alone
        return np.full((h, w), 90, np.uint8), np.full((h, w), 90, np.uint8)
    if kind == "extreme":    # the largest sums and SADs
        return np.full((h, w), 255, np.uint8), np.zeros((h, w), np.uint8)
    if kind == "period":     # many exact matches: the order decides
        t = rng.integers(0, 256, (4, 4)).astype(np.uint8)
        a = np.tile(t, (h // 4 + 1, w // 4 + 1))[:h, :w]
        return a, np.roll(a, (1, 3), (0, 1))
    ref = synth.smooth_field(w, h, seed=seed)
    return ref, synth.multi_ref_current([ref], 16, 20, seed=seed + 1)


def every_shape(w, h, seed, spread, count=2):
    rng = np.random.default_rng(seed)
    pus = []
    for part in range(25):
        pw, ph = X.PU_W[part], X.PU_H[part]
        for _ in range(count):
            x, y = int(rng.integers(0, (w - pw) // 4 + 1)) * 4, int(rng.integers(0, h - ph + 1))
            pus.append((x, y, pw, ph) + tuple(int(v) for v in rng.integers(-spread, spread + 1, 2)))
    return pus


def run(kind, w, h, pus, R, seed, n_ref=1, plain=True, oracle=True, **kw):
    kw = dict(use_fractional_me=0, **kw)
    pics = [pictures(kind, w, h, seed + 10 * r) for r in range(n_ref)]
    cur = pics[0][1]
    refs = []
    for ref, _ in pics:
        d = X.DeviceRef(w, h, frac=0)
        d.load(ref)
        refs.append(d)
    dcur = device_cur(cur)
    plan = X.Plan(X.me_params(w, h, R, LAM, **kw), X.make_pus(pus), n_ref)
    plan.run(dcur, refs)
    got = plan.fetch()
    if plain:
        other = X.Plan(X.me_params(w, h, R, LAM, **kw), X.make_pus(pus), n_ref, X.PLAN_PLAIN)
        other.run(dcur, refs)
        compare(got, other.fetch(), pus, n_ref)
    if oracle:
        exp = oracle_results(O.me_param(w, h, R, LAM, **kw), pus, cur, [oracle_ref(ref, 0) for ref, _ in pics], n_ref)
        compare(got, exp, pus, n_ref)


@pytest.mark.parametrize("R", [1, 2, 5, 8, 16, 23, 24, 31, 48, 57, 64, 65])
def test_every_shape_at_ranges_around_the_splits(R):
    run("smooth", 208, 144, every_shape(208, 144, R, 40), R, seed=R, n_ref=2)


@pytest.mark.parametrize("kind", ["noise", "flat", "extreme", "period"])
@pytest.mark.parametrize("R", [12, 33, 64])
def test_pictures_without_elimination_or_with_ties(kind, R):
    run(kind, 176, 144, every_shape(176, 144, 5 * R, 13, count=1), R, seed=3)


@pytest.mark.parametrize("kw", [dict(mv_range_x=(-40, 51), mv_range_y=(-30, 23)), dict(mv_range_x=(9, 90)),
                                dict(mv_range_y=(-77, -20))])
def test_narrow_mv_ranges(kw):
    run("smooth", 176, 144, every_shape(176, 144, 9, 60), 32, seed=6, **kw)


def test_frame_borders_and_odd_rows():
    w, h = 200, 136
    pus = [(x, y, 16, 16, 5, -7) for y in (0, 1, 119, 120) for x in (0, 4, 180, 184)]
    pus += [(136, 72, 64, 64, 0, 0), (0, 0, 64, 64, -11, 3), (192, 131, 8, 4, 2, 2), (4, 3, 32, 24, 1, 1)]
    for R in (16, 64):
        run("smooth", w, h, pus, R, seed=8)


@pytest.mark.parametrize("spread", [160, 300, 600])
def test_spread_centres_cut_the_window(spread):
    """Centres up to 150 pixels from (0, 0) on the left or above: windows in
    row ranges and cells cut into quarters and single PUs."""
    w, h = 640, 512
    rng = np.random.default_rng(spread)
    pus = [(x, y, 16, 16) + tuple(int(v) for v in rng.integers(-spread, spread + 1, 2) // (1, 4))
           for y in range(192, 320, 16) for x in range(192, 448, 16)]
    pus += [(64, 64, 64, 64, spread, 0), (448, 192, 64, 64, 0, -spread)]
    run("smooth", w, h, pus, 64, seed=4, plain=False)


def test_a_window_that_fits_without_its_sums_is_searched_exhaustively():
    """One PU whose window over both its centres (340 pixels apart) fits the
    LDS, but not with its sums: the plan is taken as ever."""
    run("smooth", 640, 192, [(64, 64, 64, 64, 1360, 0), (320, 64, 16, 16, 0, 0)], 64, seed=5, plain=False)


def test_windows_beyond_the_lds_are_refused():
    pus = X.make_pus([(256, 192, 16, 16, 1800, 0), (272, 192, 16, 16, -1800, 900), (288, 192, 16, 16, 0, -900)])
    with pytest.raises(X.XmeError, match="LDS"):
        X.Plan(X.me_params(640, 512, 64, LAM, use_fractional_me=0), pus, 1)


def test_cost_map_of_eliminated_candidates():
    """A cost map holds every candidate's cost, also those the search leaves out."""
    w, h, R = 96, 80, 24
    ref, cur = pictures("smooth", w, h, 2)
    d = X.DeviceRef(w, h, frac=0)
    d.load(ref)
    pus = [(0, 0, 16, 16, 9, 4), (64, 48, 32, 32, 0, 0), (92, 4, 4, 16, -3, 1), (40, 33, 12, 16, 0, 0)]
    prm = dict(use_fractional_me=0, mv_range_x=(-90, 77))
    plan = X.Plan(X.me_params(w, h, R, LAM, **prm), X.make_pus(pus), 1)
    cm = X.DeviceBuffer(len(pus) * 16 * R * R)
    plan.run(device_cur(cur), [d], cost_map=cm)
    maps = cm.download(len(pus) * 4 * R * R, np.int32).reshape(len(pus), 2 * R, 2 * R)
    c = O.Plane(w, h)
    c.set_picture(cur)
    for i, p in enumerate(pus):
        _, exp = O.me_search(O.me_param(w, h, R, LAM, **prm), p, c, oracle_ref(ref, 0), cost_map=True)
        assert np.array_equal(maps[i], exp), i
