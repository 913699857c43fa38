"""GPU: the 2D fused stages on blocks cut into slabs -- sides that do not
divide, slabs of one row, rows longer than a workgroup -- one RK4 step bit for
bit against the oracle, by one pool (halo gather on and off) and by a batch
of two pools of different block sizes, without and with a mask."""
import numpy as np
import pytest

from helpers import random_mask
from oracle import pyoracle as po
from wabbit_amd import lib as L
from wabbit_amd.forest import EquidistantForest
from wabbit_amd.params import ACMParams, butcher_rk4

pytestmark = pytest.mark.gpu

DT = 1e-4


def _acm(scheme, skew, masked=False):
    return ACMParams(dim=2, scheme=scheme, skew_symmetry=skew, penalization=masked, use_sponge=masked, c_0=10.0, nu=1e-3,
                     C_eta=1e-2, C_sponge=1e-2, u_mean_set=[1.0, 0.2, 0.0], domain_size=[1.0, 1.0, 1.0])


def _case(bs, scheme, skew, seed, masked=False):
    """forest, state, the oracle's state after one step"""
    g = {2: 1, 4: 3, 6: 5}[scheme]
    f = EquidistantForest(2, 2, bs, g, [1.0, 1.0])
    rng = np.random.default_rng(seed)
    u = 0.1 * rng.standard_normal((f.n, 3, 1, bs[1] + 2 * g, bs[0] + 2 * g))
    mask = random_mask(f, seed) if masked else None
    run = po.EquidistantRun(po.make_params(_acm(scheme, skew, masked)), bs, g, scheme // 2, 3, 2, [1.0, 1.0], u.copy(),
                            f.block_at(), mask)
    run.step(DT)
    return f, u, run.hvy[:, :, 0, g:g + bs[1], g:g + bs[0]]


def _pool(f, u, depth, gather, mask=None):
    p = L.Pool(2, f.bs, f.g, 3, f.n, n_work_slots=3, n_mask=0 if mask is None else 6)
    if mask is not None:
        p.upload(L.WH_MASK, 0, mask)
    p.set_tuning(L.WH_TUNE_GATHER, gather)
    p.upload(L.WH_BLOCK, 0, u)
    p.set_active(f.active, f.x0dx)
    p.set_patches(0, f.same_level_patches(depth))
    return p


def _got(p, f):
    g = f.g
    return p.download(L.WH_BLOCK, 0, f.n)[:, :, 0, g:g + f.bs[1], g:g + f.bs[0]]


CASES = [([16, 16], 4, False), ([24, 24], 6, True), ([48, 20], 4, True), ([9, 33], 6, False), ([20, 49], 2, False),
         ([130, 6], 4, False), ([260, 5], 4, True)]


@pytest.mark.parametrize("bs,scheme,skew", CASES)
def test_slabs_match_oracle(bs, scheme, skew):
    f, u, want = _case(bs, scheme, skew, 4)
    for gather in (1, 0):
        p = _pool(f, u, scheme // 2, gather)
        p.rk_step(L.acm_params_c(_acm(scheme, skew)), butcher_rk4(), 0.0, DT, 2)
        assert np.array_equal(_got(p, f), want), (bs, gather)
        p.close()


@pytest.mark.parametrize("bs,scheme,skew", CASES)
def test_masked_slabs_match_oracle(bs, scheme, skew):
    """Penalised + sponge: the mask of a thread's first point is loaded ahead,
    that of its further ones (rows longer than a workgroup) from memory.  By
    one pool and by a batch of one."""
    f, u, want = _case(bs, scheme, skew, 4, True)
    ac, mask = L.acm_params_c(_acm(scheme, skew, True)), random_mask(f, 4)
    for gather in (1, 0):
        p = _pool(f, u, scheme // 2, gather, mask)
        p.rk_step(ac, butcher_rk4(), 0.0, DT, 2)
        assert np.array_equal(_got(p, f), want), gather
        p.close()
    p = _pool(f, u, scheme // 2, 1, mask)
    p.set_block_groups(np.zeros(f.n, np.int32), 1)
    st = L.BatchStepper([p])
    st.rk_step(ac, butcher_rk4(), [DT])
    st.synchronize()
    assert np.array_equal(_got(p, f), want)
    st.close()
    p.close()


@pytest.mark.parametrize("a,b", [(0, 2), (5, 2), (6, 5)])
def test_slabs_of_a_batch(a, b):
    """Two pools with different slab counts; the constants of the first case."""
    _, scheme, skew = CASES[a]
    cases = [_case(CASES[i][0], scheme, skew, i) for i in (a, b)]
    pools = [_pool(f, u, scheme // 2, 1) for f, u, _ in cases]
    for p, (f, _, _) in zip(pools, cases):
        p.set_block_groups(np.zeros(f.n, np.int32), 1)
    st = L.BatchStepper(pools)
    st.rk_step(L.acm_params_c(_acm(scheme, skew)), butcher_rk4(), [DT, DT])
    st.synchronize()
    for p, (f, _, want) in zip(pools, cases):
        assert np.array_equal(_got(p, f), want)
    st.close()
    for p in pools:
        p.close()
