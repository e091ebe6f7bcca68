"""GPU: small PUs of the pattern searches take more lanes than their class has
while the launch stays within 2048 waves, and the candidate and sub-pel stages
pack 4 or 2 small PUs per wave.  Instance counts on both sides of the rule's
edges, and counts that leave waves partly empty, against the oracle."""
import pytest

from tests.test_gpu_me import run_case
from xavs2_amd import lib as X
from xavs2_amd import synth

pytestmark = pytest.mark.gpu


def tiling(w, h, pw, ph):
    return [(x, y, pw, ph, 0, 0) for (x, y, _, _) in synth.shape_tiling(w, h, pw, ph)]


# 8x8 instances: 2 per wave to 4096, 4 to 8192 (2048 waves), 8 to 16384, then 16
@pytest.mark.parametrize("method", [X.ME_DIA, X.ME_HEX, X.ME_TZ])
@pytest.mark.parametrize("w,h,n_ref", [(512, 256, 2), (512, 264, 2), (512, 256, 4), (512, 264, 4), (640, 512, 4)])
def test_lanes_of_small_pus(method, w, h, n_ref):
    run_case(w, h, tiling(w, h, 8, 8), 16, n_ref=n_ref, seed=method + h,
             prm_kw=dict(me_method=method, use_fractional_me=0))


# per class of the sub-pel stage: a few PUs of each size, so that the last wave of a class is partly empty
@pytest.mark.parametrize("method", [X.ME_FS, X.ME_HEX])
@pytest.mark.parametrize("counts", [(1, 0, 0, 0), (3, 1, 0, 1), (5, 3, 2, 0), (0, 7, 1, 2), (9, 2, 3, 1)])
@pytest.mark.parametrize("n_ref", [1, 3])
def test_partly_filled_waves(method, counts, n_ref):
    w, h = 256, 128
    pus = []
    for (pw, ph), n in zip([(8, 8), (16, 8), (32, 16), (64, 64)], counts):
        pus += tiling(w, h, pw, ph)[:n]
    run_case(w, h, pus, 16, n_ref=n_ref, seed=sum(counts), prm_kw=dict(me_method=method))
