"""Islands against the serial kernel in the kinds and precisions that the
oracle does not cover: the same world alone, resolved by islands, and with
bodies out of reach added up to more than the islands' tables hold, resolved by
the serial kernel.  State, contact internals, iteration counts and labels bit
for bit, with budgets that stop the world everywhere."""
import numpy as np
import pytest

from cubez_amd import World
from tests.test_gpu_islands import INTERNALS, _pile
from tests.test_gpu_left import padded

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "vel", "rot", "quat", "iit_world", "transform", "motion", "flags")
# islands of up to 64 contacts, of 65 to 256, 257 to 512 and more
CASES = [(64, 1.0, 300), (200, 1.0, 240), (250, 0.4, 150), (200, 0.5, 200)]
BUDGETS = [(4, 0), (1, 0), (2, 0), (4, 1), (4, 2), (4, 33), (4, 100), (4, 300)]


def _both(sc, precision, kind):
    worlds = [World(s, precision=precision) for s in (sc, padded(sc, 2049))]
    if kind == "materials":
        rng = np.random.default_rng(7)
        f = rng.uniform(0.0, 1.2, 2049)
        f[rng.random(2049) < 0.25] = 0.0
        e = rng.uniform(0.0, 0.5, 2049)
        for w in worlds:
            w.set_materials(True)
            w.set("friction", f[:w.n_bodies])
            w.set("restitution", e[:w.n_bodies])
    return worlds


def _equal(a, b, n, what):
    assert (a.resolver_iterations() == b.resolver_iterations()).all(), what
    for k in FIELDS:
        x, y = (w.get(k).reshape(w.n_bodies, -1)[:n] for w in (a, b))
        assert np.array_equal(x, y, equal_nan=True), (what, k)
    x, y = a.contacts(0), b.contacts(0)
    for k in INTERNALS:
        assert np.array_equal(x[k], y[k], equal_nan=True), (what, k)


@pytest.mark.parametrize("kind", ["plain", "materials", "labels"])
@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("n,squeeze,at", CASES)
def test_islands_equal_the_serial_kernel(n, squeeze, at, precision, kind):
    sc = _pile(n, squeeze)
    a, b = _both(sc, precision, kind)
    with a, b:
        for w in (a, b):
            w.step(sc.dt, at, 4)
        _equal(a, b, n, "steps")
        saved = [w.checkpoint() for w in (a, b)]
        for mult, fixed in BUDGETS:
            if kind == "labels" and fixed:
                continue
            for w, ck in zip((a, b), saved):
                w.restore(ck)
                if kind == "materials":
                    assert (w.get("friction")[:n] == a.get("friction")).all()
                w.integrate(sc.dt)
                w.narrowphase()
                if kind == "labels":
                    w.sur_reserve(8000)
                    assert w.sur_collect(sc.dt, mult) > 20
                else:
                    w.resolve(sc.dt, mult, fixed)
            _equal(a, b, n, (mult, fixed))
            if kind == "labels":
                x, y = a.sur_dataset()[1], b.sur_dataset()[1]
                assert np.array_equal(x, y) and np.abs(x).max() > 0
