"""GPU: the 3D fused stages reading whole same-level faces from the
neighbours' interiors (WH_TUNE_GATHER on a 3D pool) against the same steps
with every ghost fill launched: the whole block array, ghost nodes
included, bit for bit, on uniform and mixed-level forests and on patch
tables the gather must leave alone in part."""
import numpy as np
import pytest

from wabbit_amd import lib as L
from wabbit_amd.params import ACMParams, butcher_rk4
from wabbit_amd.tree import Forest

pytestmark = pytest.mark.gpu


def _forest(bs, g, refined):
    """64 blocks of level 2, every `refined`-th replaced by its 8 daughters (0: none)."""
    f = Forest(3, 3, bs, g, [1.0, 1.0, 1.0], 320)
    tc, lv = [], []
    for k in range(64):
        if refined and k % refined == 0:
            tc += [k * 8 + d for d in range(8)]
            lv += [3] * 8
        else:
            tc.append(k * 8)
            lv.append(2)
    ids = np.random.default_rng(3).permutation(320)[:len(tc)]
    f.set_blocks(np.array(tc, np.int64), np.array(lv, np.int32), ids.astype(np.int32))
    return f


def _overwrite(patches, bs):
    """Second-stage copies into a part of some faces, and one face filled by
    two patches instead of one: neither may be gathered."""
    whole = np.flatnonzero((patches["op"] == 0) & (patches["n"][:, 1] == bs[1]) & (patches["n"][:, 2] == bs[2]))
    extra = patches[whole[::7]].copy()
    extra["n"][:, 1], extra["stage"] = 3, 2
    extra["send"] = np.roll(extra["send"], 1)
    halves = patches[whole[3]:whole[3] + 1].copy().repeat(2)
    halves["n"][:, 2] = bs[2] // 2
    halves["recv_lo"][1, 2] += bs[2] // 2
    halves["send_lo"][1, 2] += bs[2] // 2
    return np.concatenate([np.delete(patches, whole[3]), halves, extra])


def _run(gather, bs, g, depth, scheme, skew, refined, table, ysplit, steps=2):
    f = _forest(bs, g, refined)
    patches = f.patches(depth, depth, 4)
    if table == "shuffled":
        patches = np.random.default_rng(1).permutation(patches)
    elif table == "overwritten":
        patches = _overwrite(patches, bs)
    _, _, hv, x = f.blocks()
    p = L.Pool(3, bs, g, 4, 320, n_work_slots=3)
    try:
        p.set_tuning(L.WH_TUNE_GATHER, gather)
        p.set_tuning(L.WH_TUNE_K3D_YSPLIT, ysplit)
        p.upload(L.WH_BLOCK, 0, 0.1 * np.random.default_rng(5).standard_normal((320,) + p.block_shape()))
        p.set_active(hv, x)
        p.set_patches(0, patches)
        ac = L.acm_params_c(ACMParams(dim=3, scheme=scheme, skew_symmetry=skew, penalization=False, c_0=10.0, nu=1e-3))
        for _ in range(steps):
            p.rk_step(ac, butcher_rk4(), 0.0, 1e-4, 2)
        return p.download(L.WH_BLOCK, 0, 320)
    finally:
        p.close()
        f.close()


@pytest.mark.parametrize("bs,g,depth,scheme,skew,refined,table,ysplit", [
    ([8, 8, 8], 3, 2, 4, False, 0, "plain", -1),         # uniform: no patch is left
    ([12, 16, 8], 6, 2, 4, False, 5, "plain", -1),       # mixed levels, unequal sides
    ([12, 16, 8], 6, 2, 4, False, 5, "plain", 2),        # slabs: faces in y only at the ends
    ([12, 16, 8], 6, 2, 4, True, 5, "shuffled", -1),
    ([12, 12, 12], 6, 2, 4, False, 7, "overwritten", -1),
    ([16, 16, 16], 6, 6, 4, False, 3, "plain", -1),      # patches deeper than the stencil
    ([12, 12, 12], 5, 3, 6, True, 4, "plain", -1),
    ([10, 10, 10], 3, 2, 2, False, 2, "plain", -1),
])
def test_face_gather_matches_ghost_fill(bs, g, depth, scheme, skew, refined, table, ysplit):
    on = _run(1, bs, g, depth, scheme, skew, refined, table, ysplit)
    off = _run(0, bs, g, depth, scheme, skew, refined, table, ysplit)
    print(bs, scheme, table, "max |diff|", np.abs(on - off).max(), flush=True)
    assert np.array_equal(on, off)
    assert np.all(np.isfinite(on))


@pytest.mark.parametrize("refined", [0, 5])
def test_steps_after_a_packed_step(refined):
    """The work slots are scratch after a fused step, packed on a uniform grid:
    the other paths, other stencils and a plain right-hand side on the same pool
    give what they give after a step that filled every ghost node."""
    bs, g, out = [12, 12, 12], 5, {}
    for gather in (1, 0):
        f = _forest(bs, g, refined)
        _, _, hv, x = f.blocks()
        p = L.Pool(3, bs, g, 4, 320, n_work_slots=5)
        p.set_tuning(L.WH_TUNE_GATHER, gather)
        p.upload(L.WH_BLOCK, 0, 0.1 * np.random.default_rng(5).standard_normal((320,) + p.block_shape()))
        p.set_active(hv, x)
        p.set_patches(0, f.patches(3, 3, 4))
        got = []
        for scheme, path in ((4, 2), (4, 0), (6, 2), (4, 2), (2, 1)):
            ac = L.acm_params_c(ACMParams(dim=3, scheme=scheme, penalization=False, c_0=10.0, nu=1e-3))
            p.rk_step(ac, butcher_rk4(), 0.0, 1e-4, path)
            got.append(p.download(L.WH_BLOCK, 0, 320))
        p.sync(L.WH_BLOCK, 0)
        p.rhs(ac, 0.0, L.WH_BLOCK, 1)
        got.append(p.download(L.WH_WORK + 1, 0, 320)[hv][:, :, g:-g, g:-g, g:-g])
        out[gather] = got
        p.close()
        f.close()
    for on, off in zip(out[1], out[0]):
        assert np.array_equal(on, off) and np.all(np.isfinite(on))
