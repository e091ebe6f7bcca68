"""GPU: coefficients leave the residual kernels 8 bytes a lane, four rows of
four columns exchanged between neighbouring lanes.  Where that can go wrong:
block counts around a 32x32 tile's (every remainder of a tile is a guard of its
own; nothing past the last block is written), and levels whose address is not a
multiple of 8, which take 2-byte stores."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_me import device_cur, oracle_cur, oracle_ref
from tests.test_gpu_transform import laplacian_blocks
from tests.test_oracle_recon import tiles
from xavs2_amd import lib as X
from xavs2_amd import synth

pytestmark = pytest.mark.gpu

GUARD = 0x3C3C


@pytest.mark.parametrize("n,nblk", [(4, 1), (4, 7), (4, 63), (4, 65), (8, 3), (8, 15), (8, 17), (16, 1), (16, 3),
                                    (16, 5), (32, 1), (32, 5)])
def test_block_counts_around_a_tile(n, nblk):
    blocks = laplacian_blocks(n, nblk, seed=n * 100 + nblk, zero_frac=0.2, b=20.0)
    src = X.upload(blocks)
    guard = np.full(blocks.size + 1024, GUARD, np.int16)
    lv, rc, nz = X.upload(guard), X.upload(guard), X.DeviceBuffer(4 * nblk)
    X.check(X.lib().xme_residual_batch(n, 27, 0, src.at(), lv.at(), rc.at(), nz.at(), nblk, None), "residual")
    e_level, e_recon, e_nnz = O.residual_batch(n, 27, 0, blocks)
    for buf, exp in ((lv, e_level), (rc, e_recon)):
        got = buf.download(guard.size, np.int16)
        assert np.array_equal(got[: blocks.size], exp.ravel())
        assert (got[blocks.size:] == GUARD).all()
    assert np.array_equal(nz.download(nblk, np.int32), e_nnz)


@pytest.mark.parametrize("offset", [0, 2, 4, 6, 8])
@pytest.mark.parametrize("n,frac", [(4, 2), (8, 2), (16, 2), (32, 2), (64, 2), (8, 0), (16, 0)])
def test_levels_at_any_address(n, frac, offset):
    w, h, nl = 128, 64, min(n, 32)
    ref = synth.smooth_field(w, h, seed=21)
    cur = synth.multi_ref_current([ref], 8, 8, seed=22)
    if n == 64:
        tus = np.array([[0, 0, 0, 0, 64, 64, 5, -3], [64, 0, 64, 0, 64, 64, -7, 2]], np.int32)
    else:
        tus = tiles(w, h, n, np.random.default_rng(n), far=True)
    ntu = len(tus)
    dref, dcur = X.DeviceRef(w, h, frac=frac), device_cur(cur)
    dref.load(ref)
    size = ntu * nl * nl
    level = X.upload(np.full(size + 64, GUARD, np.int16))
    rec = X.DevicePlane(w, h, pad=0, stride=dcur.stride)
    resid, rres, nnz, ssd = (X.DeviceBuffer(k) for k in (2 * ntu * n * n, 2 * ntu * n * n, 4 * ntu, 4 * ntu))
    rd, d_tus = dref.desc(), X.upload(np.ascontiguousarray(tus, np.int32))
    staged = frac == 0
    X.check(X.lib().xme_inter_recon_batch(n, 30, C.c_void_p(dcur.origin), dcur.stride, C.byref(rd), w, h,
                                          d_tus.at(), ntu,
                                          resid.at() if staged else None, level.at(offset),
                                          rres.at() if staged else None, C.c_void_p(rec.origin), rec.stride,
                                          nnz.at(), ssd.at(), None), "xme_inter_recon_batch")
    X.check(X.lib().xme_stream_sync(None), "sync")
    exp = O.inter_recon_batch(n, 30, oracle_cur(cur), oracle_ref(ref, 2), w, h, tus)
    got = level.download(size + 64, np.int16)
    k = offset // 2
    assert np.array_equal(got[k: k + size], np.asarray(exp[0]).ravel())
    assert (got[:k] == GUARD).all() and (got[k + size:] == GUARD).all()
    assert np.array_equal(nnz.download(ntu, np.int32), exp[2])
