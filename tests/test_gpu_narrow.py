"""Launches of so many worlds that each gets half a workgroup's threads, with
some worlds left to whole workgroups: the same worlds in a small launch, bit for
bit."""
import numpy as np
import pytest

from cubez_amd import World, scenes
from tests.test_gpu_islands import _island_sizes, _pile

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "vel", "rot", "quat", "motion")


# the line is 2048 worlds in FP64, 3072 in FP32
@pytest.mark.parametrize("precision,worlds", [("f64", 2049), ("f32", 3073)])
@pytest.mark.parametrize("mult,fixed", [(4, 0), (1, 0), (4, 300), (4, 12)])
def test_worlds_of_large_launches(precision, worlds, mult, fixed):
    small = scenes.batched(4, 1, 12, 12)
    small.fields["pos"] *= (0.4, 0.1, 0.4)
    kinds = [_pile(400, 0.4), _pile(24, 1.0), _pile(120, 0.4), small]
    of = np.full(worlds, 3)
    of[[3, 1000, worlds - 1]] = 1
    of[[7, 500, worlds - 2]] = 2
    of[[0, 700]] = 0
    off = np.cumsum([0] + [k.n_bodies for k in kinds])
    body = np.concatenate([np.arange(off[k], off[k + 1]) for k in of])
    with World(scenes.concat(kinds), precision=precision) as a, \
            World(scenes.concat([kinds[k] for k in of]), precision=precision) as b:
        largest = 0
        for _ in range(3):
            for w in (a, b):
                w.step(small.dt, 70, 4)
                w.integrate(small.dt)
                w.narrowphase()
                w.resolve(small.dt, mult, fixed)
            assert (b.contact_counts() == a.contact_counts()[of]).all()
            assert (b.resolver_iterations() == a.resolver_iterations()[of]).all()
            for f in FIELDS:
                x, y = (w.get(f).reshape(w.n_bodies, -1) for w in (a, b))
                assert np.array_equal(y, x[body], equal_nan=True), f
            cs = a.contacts(0)
            if len(cs["body0"]):
                largest = max(largest, _island_sizes(kinds[0].n_bodies, cs).max())
        assert largest > 1024  # more than half a workgroup's tables hold
