"""GPU: host-built lists and reduction results around the sizes up to which
kernels read and write them in host memory, and the maxima over columns that
end inside a group of loads; against the same operations in numpy, exactly."""
import numpy as np
import pytest

from wabbit_amd import lib as L
from wabbit_amd import wavelets as W

pytestmark = pytest.mark.gpu


def wavelet_pool(dim, bs, neq, nb, name="CDF22"):
    w = W.setup(name)
    pool = L.Pool(dim, bs, w.g, neq, nb, n_work_slots=2, n_tmp_eqn=neq)
    W.set_wavelet(pool, w)
    return pool, w.g


def details(u, g, dim):
    """max |v| over the interior without the points even in every direction"""
    a = np.abs(u[(Ellipsis,) + (slice(g, -g),) * dim])
    a[(Ellipsis,) + (slice(None, None, 2),) * dim] = 0.0
    return a.max(axis=tuple(range(-dim, 0)))


# 512 ids are 2 KB; 10922 and 10923 blocks of 3 components lie at 256 KB of results
@pytest.mark.parametrize("n", [1, 512, 513, 10922, 10923])
def test_details_of_listed_blocks(n):
    pool, g = wavelet_pool(2, [6, 6, 1], 3, n)
    rng = np.random.default_rng(n)
    u = rng.standard_normal((n, 3, 1, 6 + 2 * g, 6 + 2 * g))
    pool.upload(L.WH_BLOCK, 0, u)
    want = details(u, g, 2).reshape(n, 3)
    ids = rng.permutation(n).astype(np.int32)
    for _ in range(3):  # the same space again, other blocks in it
        assert np.array_equal(W.detail_blocks(pool, L.WH_BLOCK, ids, [1, 1, 1], 3), want[ids])
        ids = ids[::-1].copy()
    flags, detail = W.fwt_threshold(pool, L.WH_BLOCK, L.WH_TMP, ids, [2.0] * 3, [1, 1, 1])
    wc = details(pool.download(L.WH_TMP, 0, n).reshape(u.shape), g, 2).reshape(n, 3)[ids]
    assert np.array_equal(detail, wc)
    assert np.array_equal(np.asarray(flags), np.where((wc <= 2.0).all(axis=1), -1, 0))
    pool.close()


@pytest.mark.parametrize("bs", [[6, 8, 4], [8, 6, 10], [10, 18, 24]])
def test_details_of_3d_columns(bs):
    n = 5
    pool, g = wavelet_pool(3, bs, 2, n)
    u = np.random.default_rng(3).standard_normal((n, 2) + tuple(b + 2 * g for b in bs[::-1]))
    pool.upload(L.WH_BLOCK, 0, u)
    got = W.detail_blocks(pool, L.WH_BLOCK, np.arange(n), [1, 2], 2)
    assert np.array_equal(got, details(u, g, 3))
    pool.close()


# 18724 records of 56 bytes are the last list within 1 MB
@pytest.mark.parametrize("npatch", [18724, 18725])
def test_patch_lists(npatch):
    bs, nb = 8, 240
    pool, g = wavelet_pool(2, [bs, bs, 1], 1, nb)
    m = bs + 2 * g
    rng = np.random.default_rng(5)
    u = rng.standard_normal((nb, 1, 1, m, m))
    pool.upload(L.WH_BLOCK, 0, u)
    ghost = [(x, y) for y in range(m) for x in range(m) if not (g <= x < g + bs and g <= y < g + bs)]
    assert len(ghost) * nb >= npatch
    p = np.zeros(npatch, L.PATCH_DTYPE)
    k = np.arange(npatch)
    p["recv"], p["send"] = k % nb, rng.integers(0, nb, npatch)
    xy = np.array(ghost)[k // nb]
    p["recv_lo"][:, :2], p["send_lo"][:, :2] = xy, rng.integers(g, g + bs, (npatch, 2))
    p["n"], p["op"], p["stage"] = 1, L.WH_PATCH_COPY, 1
    W.run_patches(pool, L.WH_BLOCK, p)
    want = u.copy()
    want[p["recv"], 0, 0, xy[:, 1], xy[:, 0]] = u[p["send"], 0, 0, p["send_lo"][:, 1], p["send_lo"][:, 0]]
    assert np.array_equal(pool.download(L.WH_BLOCK, 0, nb).reshape(u.shape), want)
    pool.close()


# boxes of 32 bytes: 32768 lie within 1 MB, their maxima within 256 KB
@pytest.mark.parametrize("n", [1, 32768, 32769])
def test_box_maxima(n):
    pool, g = wavelet_pool(2, [4, 4, 1], 1, n)
    m = 4 + 2 * g
    u = np.random.default_rng(7).standard_normal((n, 1, 1, m, m))
    pool.upload(L.WH_BLOCK, 0, u)
    want = np.abs(u[..., g:-g, g:-g]).max()
    assert W.component_norm(pool, L.WH_BLOCK, np.arange(n), np.zeros(n), [1], 1, 0, [1.0, 1.0])[0] == want
    pool.close()
