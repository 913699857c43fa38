"""GPU: the 3D transforms of many blocks, which run in one sweep over z
(few blocks take the plane and column kernels of the other wavelet tests),
and adapt_tree on as many, against the oracle bit for bit."""
import numpy as np
import pytest

from helpers import smooth_blocks
from oracle import pyoracle as po
from wabbit_amd import lib as L
from wabbit_amd import wavelets as W
from wabbit_amd.forest import equidistant_treecodes
from wabbit_amd.tree import Forest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wav,bs,n", [("CDF40", 12, 520), ("CDF42", 14, 520), ("CDF44", 12, 515), ("CDF44", 20, 513),
                                      ("CDF62", 12, 520), ("CDF60", 12, 512), ("CDF22", 12, 520)])
def test_transforms_of_many_blocks(wav, bs, n):
    w, wo = W.setup(wav), po.wavelet(wav)
    g, neq, kinds = w.g, 2, 5
    rng = np.random.default_rng(2)
    one = (kinds, neq) + (bs + 2 * g,) * 3
    src, prior = rng.standard_normal(one), rng.standard_normal(one)
    kind = rng.integers(0, kinds, n)
    pool = L.Pool(3, [bs] * 3, g, neq, n, n_work_slots=2, n_tmp_eqn=neq)
    W.set_wavelet(pool, w)
    ids = rng.permutation(n).astype(np.int32)
    for fn, ofn in ((W.fwt_blocks, po.fwt_block), (W.iwt_blocks, po.iwt_block)):
        pool.upload(L.WH_TMP, 0, src[kind])
        pool.upload(L.WH_BLOCK, 0, prior[kind])
        fn(pool, L.WH_TMP, L.WH_BLOCK, ids)
        want = np.stack([ofn(wo, 3, [bs] * 3, g, src[k], prior[k]) for k in range(kinds)])
        assert np.array_equal(pool.download(L.WH_BLOCK, 0, n), want[kind])
        assert np.array_equal(pool.download(L.WH_TMP, 0, n), src[kind])
    pool.close()


@pytest.mark.parametrize("wav,bs", [("CDF44", 16), ("CDF40", 8)])
def test_adapt_many_blocks(wav, bs):
    """512 leaves on one level: the decomposition copies and transforms them
    in one launch, in place."""
    w = W.setup(wav)
    g, neq, jmin, jmax, eps = w.g, 2, 1, 3, 3e-2
    tcs, lev = equidistant_treecodes(3, 3, jmax)
    n = len(tcs)
    hvy = smooth_blocks(tcs, lev, jmax, 3, bs, g, 4, neq)
    t = po.Tree(po.wavelet(wav), 3, jmin, jmax, [bs] * 3, g, tcs, lev, hvy, indicator=1, eps=eps, groups=[1, 1])
    t.sync()
    t.adapt()
    tco, lvo, hvo = t.get()
    t.close()
    f = Forest(3, jmax, [bs] * 3, g, [1.0] * 3, nb_max=2 * n)
    f.set_blocks(tcs, lev, np.arange(n, dtype=np.int32))
    pool = L.Pool(3, [bs] * 3, g, neq, 2 * n, n_work_slots=2, n_tmp_eqn=neq)
    W.set_wavelet(pool, w)
    pool.upload(L.WH_BLOCK, 0, hvy)
    W.sync_tree(pool, f)
    W.adapt_tree(pool, f, W.adapt_params(jmin, jmax, W.WH_IND_THRESHOLD, use_ce=bool(w.lifted), eps=eps, groups=[1, 1]))
    tc, lv, hv, _ = f.blocks()
    key = {(int(a), int(b)): int(h) for a, b, h in zip(tc, lv, hv)}
    assert sorted(key) == sorted((int(a), int(b)) for a, b in zip(tco, lvo))
    print(wav, n, "->", len(tco), "leaves", flush=True)
    all_blocks = pool.download(L.WH_BLOCK, 0, 2 * n)
    assert np.array_equal(np.stack([all_blocks[key[(int(a), int(b))]] for a, b in zip(tco, lvo)]), hvo)
    pool.close()
    f.close()
