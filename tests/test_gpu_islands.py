"""The resolver by islands against the oracle, bit for bit, where it can go
wrong: islands of every size class (their limits are 4, 8, 16, 32, 64, 256 and
512 contacts), a world's islands of more than 64 contacts together, iteration
budgets that stop a world in the middle (before any island is done, while the
largest one runs, between equal keys), worlds of more bodies than the kernel's
tables hold, and a log pool too small for every world over its budget."""
import numpy as np
import pytest
from scipy.sparse import coo_matrix
from scipy.sparse.csgraph import connected_components

from cubez_amd import World, scenes
from oracle.cbz_oracle import OracleWorld
from tests.test_gpu_parity import assert_state_equal, same

pytestmark = pytest.mark.gpu

INTERNALS = ("pen", "cvel", "ddv", "c2w", "rel")


def _pile(n, squeeze, seed=5):
    sc = scenes.cubedrop(seed, n)
    sc.fields["pos"][:, 0] *= squeeze
    sc.fields["pos"][:, 2] *= squeeze
    return sc


def _island_sizes(n, cs):
    m = cs["body1"] >= 0
    g = coo_matrix((np.ones(m.sum()), (cs["body0"][m], cs["body1"][m])), shape=(n, n))
    lab = connected_components(g, directed=False)[1][cs["body0"]]
    return np.bincount(lab)[np.unique(lab)]


def _resolve_both(w, worlds, dt, mult=4, fixed=0):
    """Integrate, narrowphase and resolve on both sides; everything equal."""
    w.integrate(dt)
    w.narrowphase()
    w.resolve(dt, mult, fixed)
    it = w.resolver_iterations()
    sizes = []
    for wi, o in enumerate(worlds):
        o.integrate(dt)
        cs = o.narrowphase()
        sizes.append(_island_sizes(o.n, cs))
        before = dict(o.counters())
        out = o.resolve(cs, dt, fixed or mult * len(cs))
        after = o.counters()
        used = (after["pos_iters"] - before["pos_iters"], after["vel_iters"] - before["vel_iters"])
        if mult or fixed:  # without a budget, the counts of the resolve before stay
            assert tuple(it[wi]) == used, (wi, it[wi], used)
        gc = w.contacts(wi)
        for k in INTERNALS:
            assert same(gc[k], out[k]), (wi, k)
        assert_state_equal(w, o, o.body0, o.n)
    return np.concatenate(sizes), it


# (cubes, squeeze of the floor, step): the largest island falls into the class
@pytest.mark.parametrize("n,squeeze,at,lo,hi", [
    (64, 1.0, 300, 9, 16), (200, 1.0, 200, 33, 64), (200, 1.0, 240, 65, 256), (120, 0.3, 200, 129, 256),
    (200, 0.5, 200, 513, 2048), (250, 0.4, 150, 257, 512)])
def test_island_classes(n, squeeze, at, lo, hi):
    sc = _pile(n, squeeze)
    o = OracleWorld(sc)
    o.calculate_derived()
    with World(sc) as w:
        w.step(sc.dt, at, 4)
        o.step(sc.dt, at, 4)
        sizes, _ = _resolve_both(w, [o], sc.dt)
        assert lo <= sizes.max() <= hi, sizes.max()
        _resolve_both(w, [o], sc.dt)


# budgets: none, one, a few, inside the position phase, inside the velocity
# phase with and without a big island
@pytest.mark.parametrize("n,squeeze,at", [(64, 1.0, 300), (200, 1.0, 240), (200, 0.5, 200)])
@pytest.mark.parametrize("mult,fixed", [(0, 0), (4, 1), (4, 2), (4, 33), (4, 100), (1, 0), (2, 0)])
def test_budget_stops_the_world_where_the_serial_loop_stops(n, squeeze, at, mult, fixed):
    sc = _pile(n, squeeze)
    o = OracleWorld(sc)
    o.calculate_derived()
    with World(sc) as w:
        w.step(sc.dt, at, 4)
        o.step(sc.dt, at, 4)
        _resolve_both(w, [o], sc.dt, mult, fixed)


@pytest.mark.parametrize("small_pool", [False, True])
def test_towers_over_their_budget(small_pool):
    """Every world of standing towers exceeds its budget in the first step,
    with equal keys everywhere; with as many contact slots as contacts the log
    pool runs out and the rest of the worlds take the serial kernel."""
    sc = scenes.towers(0, 64)
    worlds = [OracleWorld(sc, k) for k in range(sc.n_worlds)]
    for o in worlds:
        o.calculate_derived()
    with World(sc) as w:
        w.integrate(sc.dt)
        n = w.narrowphase()
    with World(sc, contact_capacity=n + 64 if small_pool else 0) as w:
        _, it = _resolve_both(w, worlds, sc.dt)
        counts = w.contact_counts()
    assert (it[:, 1] == 4 * counts).all()
    assert n * 13 > 65536  # 17 iterations per contact against 4 log slots


@pytest.mark.parametrize("n", [2048, 2049])
def test_world_of_more_bodies_than_the_tables_hold(n):
    sc = scenes.batched(11, 1, n, n)
    sc.fields["pos"][:, 1] = 0.8 + 0.9 * np.arange(n) / n
    o = OracleWorld(sc)
    o.calculate_derived()
    with World(sc) as w:
        _resolve_both(w, [o], sc.dt)
