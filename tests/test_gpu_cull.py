"""The narrowphase's cull and pair test where their rules turn: worlds up to
and past one task per wave, shapes of every kind, bodies far from the origin
(the FP32 test's margin), touching its bound, and non-finite."""
import numpy as np
import pytest

from cubez_amd import World, scenes
from tests.test_gpu_broadphase import FIELDS
from tests.test_gpu_parity import same

pytestmark = pytest.mark.gpu


def _against_list(sc, pos=None, precision="f64"):
    """All-pairs contacts against the same pairs as an explicit list in the
    emission order, which no cull touches."""
    one, two = [], []
    for w in range(sc.n_worlds):
        b0, b1 = int(sc.body_off[w]), int(sc.body_off[w + 1])
        for i in range(b0, b1):
            for k in range(int(sc.plane_off[w]), int(sc.plane_off[w + 1])):
                one.append(i), two.append(-(k + 1))
            for j in range(b0, b1):
                if j != i:
                    one.append(i), two.append(j)
    with World(sc, precision=precision, contact_capacity=200_000) as w:
        if pos is not None:
            w.set("pos", pos)
        w.calculate_derived()
        total = w.narrowphase()
        got = w.contacts(-1, internals=False)
        assert w.narrowphase_pairs(np.array(one, np.int32), np.array(two, np.int32)) == total
        want = w.contacts(-1, internals=False)
    for f in FIELDS:
        assert same(got[f], want[f]), f
    return total


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("shift", [0.0, 1.0e4, 1.0e7])
def test_cull_of_mixed_shapes_far_from_the_origin(precision, shift):
    sc = scenes.ballistic(3, 70, 75)
    rng = np.random.default_rng(int(shift) % 97)
    pos = sc.fields["pos"].copy()
    pos[:, :] = rng.uniform(-9, 9, pos.shape)
    pos[5:60] = pos[5] + rng.normal(0, 1.5, (55, 3))  # a dense clump
    pos[:, 0] += shift
    pos[:, 1] += 4.0
    assert _against_list(sc, pos, precision) > 100


def test_cull_at_its_bound_and_non_finite():
    sc = scenes.cubedrop(1, 130)  # two full column tiles and a ragged one
    n = sc.n_bodies
    r = np.linalg.norm(sc.fields["half"], axis=1)
    pos = np.zeros((n, 3))
    # a chain in which each next body sits within rounding of the bound of the last
    step = np.sqrt(3.003) * (r[1:] + r[:-1]) * (1 + np.linspace(-1e-7, 1e-7, n - 1))
    pos[1:, 0] = np.cumsum(step)
    pos[:, 1] = 5.0
    _against_list(sc, pos)
    pos[:, 0] %= 7.0
    pos[3] = np.nan
    pos[64, 1] = np.inf
    pos[128, 2] = -np.inf
    assert _against_list(sc, pos) > 0


def test_cull_of_small_worlds_and_of_many_tasks():
    """600 worlds of 1 to 33 bodies, and 480 of 90 to 140: more tasks than waves
    that fit the chip at once."""
    sc = scenes.batched(11, 600, 1, 33)
    pos = sc.fields["pos"].copy()
    pos[:, 1] = 1.0 + (pos[:, 1] % 5.0)
    assert _against_list(sc, pos) > 0
    sc = scenes.batched(12, 480, 90, 140)  # too many pairs for a list: the broadphase's contacts
    n, planes = np.diff(sc.body_off), np.diff(sc.plane_off)
    assert int(np.sum(-(-(n + planes) // 64) * -(-n // 16))) > 8192
    with World(sc) as w:
        w.step(sc.dt, 100, 4)
        w.integrate(sc.dt)
        total = w.narrowphase()
        a = w.contacts(-1, internals=False)
        assert w.narrowphase_broad()[0] == total > 0
        b = w.contacts(-1, internals=False)
    for f in FIELDS:
        assert same(a[f], b[f]), f
