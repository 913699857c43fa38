"""GPU: the block dt's minimum in one launch that ends with the clamps and the
time advance -- fewer blocks than a workgroup takes, more than the launch has
workgroups, wavefront and workgroup blocks -- against the oracle's block dt,
bit for bit, between replayed steps that use the same accumulator."""
import numpy as np
import pytest

from oracle import pyoracle as po
from wabbit_amd import lib as L
from wabbit_amd.forest import EquidistantForest
from wabbit_amd.params import ACMParams, TimeParams, butcher_rk4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,bs,n", [(2, 8, 1), (2, 8, 3), (2, 24, 5), (2, 8, 1100), (2, 26, 600), (3, 8, 2), (3, 6, 700)])
def test_dt_of_many_and_few_blocks(dim, bs, n):
    g = 3
    acm = ACMParams(dim=dim, scheme=4, penalization=False, c_0=10.0, nu=1e-4)
    rng = np.random.default_rng(n)
    p = L.Pool(dim, [bs] * dim, g, dim + 1, n, n_work_slots=0)
    u = rng.standard_normal((n,) + p.block_shape()) * rng.uniform(0.1, 5.0, (n, 1, 1, 1, 1))
    p.upload(L.WH_BLOCK, 0, u)
    x = np.zeros((n, 6))
    x[:, 3:] = rng.uniform(0.5, 2.0, (n, 1)) * 0.01
    act, xs = rng.permutation(n), x
    p.set_active(act, xs)
    op = po.make_params(acm)
    want = min(po.dt_block(op, [bs] * dim, g, xs[k, 3:3 + dim], u[b]) for k, b in enumerate(act))
    for _ in range(3):
        assert p.dt(L.acm_params_c(acm)) == want
    p.set_active([], np.zeros((0, 6)))
    assert p.dt(L.acm_params_c(acm)) == 9.0e9
    p.set_active(act, xs)
    assert p.dt(L.acm_params_c(acm)) == want
    p.close()


def test_dt_between_replayed_steps():
    f = EquidistantForest(2, 3, [16, 16], 3, [1.0, 1.0])
    acm = L.acm_params_c(ACMParams(dim=2, scheme=4, penalization=False, c_0=20.0, nu=1e-3, CFL=0.5))
    tp = L.time_params_c(TimeParams(time_max=1e9))
    p = L.Pool(2, [16, 16], 3, 3, f.n, n_work_slots=3)
    p.upload(L.WH_BLOCK, 0, 0.2 * np.random.default_rng(1).standard_normal((f.n,) + p.block_shape()))
    p.set_active(f.active, f.x0dx)
    p.set_patches(0, f.same_level_patches(2))
    p.time_set(0.5, 7)
    time, it = 0.5, 7
    for n in (1, 1, 3, 1):
        first = p.dt(acm)
        p.run_steps(acm, butcher_rk4(), tp, n, use_graph=True)
        t, i, last = p.time_get()
        if n == 1:
            assert last == first and t == time + first
        assert i == it + n and t > time
        time, it = t, i
    # a step at the stop time takes no dt
    p.run_steps(acm, butcher_rk4(), L.time_params_c(TimeParams(time_max=time)), 1, use_graph=False)
    assert p.time_get() == (time, it, 0.0)
    p.close()


@pytest.mark.parametrize("use_graph", [False, True])
def test_refused_step_leaves_the_time(use_graph):
    """A block whose tile the 2D stages refuse: time, iteration and state stay,
    and the pool's next step starts from them."""
    bs, g = 96, 2
    f = EquidistantForest(2, 1, [bs, bs], g, [1.0, 1.0])
    acm = L.acm_params_c(ACMParams(dim=2, scheme=4, penalization=False, c_0=20.0, nu=1e-3, CFL=0.5))
    p = L.Pool(2, [bs, bs], g, 3, f.n, n_work_slots=3)
    u = 0.2 * np.random.default_rng(1).standard_normal((f.n,) + p.block_shape())
    p.upload(L.WH_BLOCK, 0, u)
    p.set_active(f.active, f.x0dx)
    p.set_patches(0, f.same_level_patches(2))
    p.time_set(0.5, 7)
    with pytest.raises(L.WabbitHipError) as ei:
        p.run_steps(acm, butcher_rk4(), L.time_params_c(TimeParams(time_max=1e9)), 2, use_graph=use_graph)
    assert ei.value.code == L.WH_E_ARG
    assert p.time_get() == (0.5, 7, 0.0)
    got = p.download(L.WH_BLOCK, 0, f.n)[:, :, 0, g:g + bs, g:g + bs]
    assert np.array_equal(got, u[:, :, 0, g:g + bs, g:g + bs])
    p.close()
