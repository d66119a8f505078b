"""Downloads in pieces of the one-megabyte stage: fields and contacts around
the sizes at which a second piece starts."""
import numpy as np
import pytest

from cubez_amd import World, scenes
from tests.test_gpu_parity import same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("worlds", [5460, 5461, 5462, 10923])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_fields_come_back_as_they_went(worlds, precision):
    """8 bodies per world: three planes of reals fill the stage at 43688
    (FP64: 5461 worlds) and 87376 bodies (FP32: 10922)."""
    sc = scenes.batched(0, worlds, 8, 8)
    rng = np.random.default_rng(worlds)
    with World(sc, precision=precision) as w:
        for name in ("pos", "quat", "vel", "inv_mass"):
            x = rng.normal(0, 1, w.get(name).shape).astype(np.float32).astype(np.float64)
            w.set(name, x)
            assert same(w.get(name), x), name
        fl = rng.integers(0, 2, sc.n_bodies).astype(np.uint8)
        w.set("flags", fl)
        assert np.array_equal(w.get("flags"), fl)
        assert np.array_equal(w.get("shape"), sc.fields["shape"])


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_contacts_of_all_worlds_equal_each_world_s(precision):
    """More contacts than one piece holds (5 KB per 24 contacts with every
    internal), worlds one by one against all at once."""
    sc = scenes.batched(6, 300, 8, 120)
    with World(sc, precision=precision) as w:
        w.step(sc.dt, 120, 4)
        w.integrate(sc.dt)
        assert w.narrowphase() > 12_000
        w.resolve(sc.dt, 4)
        every = w.contacts(-1)
        each = [w.contacts(k) for k in range(sc.n_worlds)]
        for name, x in every.items():
            assert same(x, np.concatenate([e[name] for e in each])), name


# FP64: 4847 contacts fill the stage with every plane; half of it holds 7280 of
# nine planes, 21840 of three; from 131073 the penetrations and from 262145 the body
# indices exceed it
@pytest.mark.parametrize("n", [4847, 4848, 4849, 7281, 14561, 21841, 43681, 131072, 131073, 262145])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_contacts_come_back_as_they_went(n, precision):
    sc = scenes.batched(0, 2, 8, 8)
    rng = np.random.default_rng(n)
    body = rng.integers(0, 16, (2, n)).astype(np.int32)
    point, normal, pen = (rng.normal(0, 1, (n, k)).astype(np.float32).astype(np.float64) for k in (3, 3, 1))
    with World(sc, precision=precision, contact_capacity=n + 3) as w:
        w.set_contacts([n - 1, 1], body[0], body[1], point, normal, pen[:, 0])
        got = w.contacts(-1)
        for name, x in (("body0", body[0]), ("body1", body[1])):
            assert np.array_equal(got[name], x), name
        for name, x in (("point", point), ("normal", normal), ("pen", pen[:, 0])):
            assert same(got[name], x), name
        one = w.contacts(1)
        assert same(one["point"], point[n - 1:]) and one["body0"][0] == body[0, -1]


# a list of 130 053 pairs and its tables are the most the stage holds
@pytest.mark.parametrize("n", [130_053, 130_054, 200_003])
def test_pair_lists_around_the_stage(n):
    sc = scenes.batched(3, 1, 200, 200)
    sc.fields["pos"][:, 1] *= 0.2
    rng = np.random.default_rng(n)
    one = rng.integers(0, 200, n).astype(np.int32)
    two = ((one + rng.integers(0, 200, n)) % 200).astype(np.int32)
    two[two == one] = -1
    with World(sc, contact_capacity=8 * n) as w:
        w.calculate_derived()
        total = w.narrowphase_pairs(one, two)
        got, parts = w.contacts(-1, internals=False), []
        counts = w.pair_contact_counts(n)
        assert total == counts.sum() > 0
        for k in range(0, n, 50_000):
            assert w.narrowphase_pairs(one[k:k + 50_000], two[k:k + 50_000]) == counts[k:k + 50_000].sum()
            parts.append(w.contacts(-1, internals=False))
        for name, x in got.items():
            assert same(x, np.concatenate([p[name] for p in parts])), name
