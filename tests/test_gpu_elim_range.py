"""GPU parity of the batched full search (successive elimination) with the
oracle and the plain plan where the best match lies just outside the search
range: candidate columns that a row of lanes has beyond 2R, the rows after the
last one of a window that is cut in row ranges, and costs near the largest."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_me import LAM, compare, device_cur, oracle_ref, oracle_results
from xavs2_amd import lib as X

pytestmark = pytest.mark.gpu


def check(ref, cur, pus, R, lam=LAM, plain=True, **kw):
    """The batched plan's results, equal to the oracle's (and the plain plan's)."""
    h, w = ref.shape
    kw = dict(use_fractional_me=0, **kw)
    dref = X.DeviceRef(w, h, frac=0)
    dref.load(ref)
    dcur = device_cur(cur)
    plan = X.Plan(X.me_params(w, h, R, lam, **kw), X.make_pus(pus), 1)
    plan.run(dcur, [dref])
    got = plan.fetch()
    compare(got, oracle_results(O.me_param(w, h, R, lam, **kw), pus, cur, [oracle_ref(ref, 0)], 1), pus, 1)
    if plain:
        other = X.Plan(X.me_params(w, h, R, lam, **kw), X.make_pus(pus), 1, X.PLAN_PLAIN)
        other.run(dcur, [dref])
        compare(got, other.fetch(), pus, 1)
    return got


@pytest.mark.parametrize("pw,ph", [(8, 8), (16, 4), (4, 16), (8, 4), (4, 8), (4, 4), (16, 16), (32, 32)])
@pytest.mark.parametrize("R", [33, 34, 40, 46, 48, 57])
def test_best_match_right_of_the_range(R, pw, ph):
    """The columns of a row of lanes end at 64 or 128, those of the range at 2R.
    Every row of these pictures is the same, and each PU matches exactly at the
    first column after the range, or at one that a row of 16 lanes wholly
    outside it starts with."""
    w, h = 384, 192
    for dx in sorted({R, R + 2, 96 - R, 97 - R}):
        if dx < R:
            continue
        row = np.random.default_rng(dx).integers(0, 256, w + 128).astype(np.uint8)
        ref, cur = np.tile(row[:w], (h, 1)), np.tile(row[dx:dx + w], (h, 1))
        pus = [(x, y, pw, ph, 0, 0) for y in (64, 96) for x in range(64, 224, 32)]
        got = check(ref, cur, pus, R, plain=False)
        assert (got["bmv_x"] < 4 * R).all()


@pytest.mark.parametrize("at", ["mvp", "origin"])
@pytest.mark.parametrize("R", [18, 17, 19, 22, 23])
def test_best_match_below_a_range_cut_in_rows(R, at):
    """A PU whose two possible centres are 240 pixels apart is searched in row
    ranges; at R = 18 the last one is the single row 35."""
    w, h, x, y, mvp = 640, 512, 400, 300, (-240, -113)
    rng = np.random.default_rng(R)
    ref, cur = (rng.integers(0, 256, (h, w)).astype(np.uint8) for _ in range(2))
    cx, cy = (x + mvp[0], y + mvp[1]) if at == "mvp" else (x, y)
    block = cur[y:y + 16, x:x + 16] // 2
    cur[y:y + 16, x:x + 16] = block
    ref[cy:cy + 16, cx:cx + 16] = block + 2                     # the better candidate: the search centre
    for dy in (R, R + 2):
        r = ref.copy()
        r[cy + dy:cy + dy + 16, cx + 5:cx + 21] = block         # an exact match outside the range
        got = check(r, cur, [(x, y, 16, 16, 4 * mvp[0], 4 * mvp[1])], R)
        assert (got["bmv_y"] < 4 * (cy - y + R)).all()


@pytest.mark.parametrize("R", list(range(1, 65)))
def test_every_range_with_cut_windows(R):
    w, h = 640, 512
    rng = np.random.default_rng(100 + R)
    ref = rng.integers(0, 256, (h, w)).astype(np.uint8)
    cur = np.roll(ref, (5, 3), (0, 1)) ^ rng.integers(0, 8, (h, w)).astype(np.uint8)
    pus = [(400, 300, 16, 16, -960, -452), (320, 64, 8, 8, -600, 700), (192, 192, 12, 16, 33, -900),
           (448, 400, 32, 32, -700, -400), (256, 256, 64, 64, 40, -24)]
    check(ref, cur, pus, R, plain=False)


@pytest.mark.parametrize("R", [24, 40, 48])
def test_largest_costs(R):
    """64x64 PUs, white against black, at the largest lambda and far from their
    MVP: every candidate costs 1044476 + 12799, the origin's as much and the
    clipped MVP's 4 more.  Nothing is eliminated, and the columns right of the
    range hold cheaper pixels."""
    w, h, x, y = 256, 256, 64, 64
    cur = np.full((h, w), 255, np.uint8)
    ref = np.zeros((h, w), np.uint8)
    # one pixel of 4 in every block at a displacement of the range, none in
    # the block one column and row before it
    for px in (x + 63 - R, x + 127 - R):
        for py in (y + 63 - R, y + 127 - R):
            ref[py, px] = 4
    ref[:, x + 63 + R:] = 100                                   # seen from displacement R on
    m = -4 * (R + 7)                                            # the window starts at -(R + 1)
    pus = [(x, y, 64, 64, -3000 - 2 * i, -3000 + 2 * i) for i in range(48)]
    got = check(ref, cur, pus, R, lam=(1 << 24) - 1, plain=False, mv_range_x=(m, 4 * (R + 60)), mv_range_y=(m, 4 * (R + 60)))
    assert (got["bmv_x"] == 0).all() and (got["bmv_y"] == 0).all()
