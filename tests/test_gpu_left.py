"""Worlds that the island kernel leaves to the serial one (more bodies than its
tables hold): more of them than the serial kernel's smallest grid, each
against the oracle."""
import numpy as np
import pytest

from cubez_amd import World, scenes
from oracle.cbz_oracle import OracleWorld
from tests.test_gpu_parity import same

pytestmark = pytest.mark.gpu


def padded(sc, total):
    """A one-world scene with bodies added up to `total`, out of reach of the
    others and of each other."""
    more = scenes.batched(9, 1, total - sc.n_bodies, total - sc.n_bodies)
    more.fields["pos"][:, 0] = 4000.0 + 8.0 * np.arange(more.n_bodies)
    more.fields["pos"][:, 1] += 5000.0
    return scenes.Scene(np.array([0, total], np.int32), sc.plane_off, sc.plane_normal, sc.plane_offset,
                        {k: np.concatenate([v, more.fields[k]]) for k, v in sc.fields.items()}, dt=sc.dt,
                        iter_mult=sc.iter_mult)


@pytest.mark.parametrize("worlds", [1, 255, 300])
def test_every_left_world_is_resolved(worlds):
    small = scenes.batched(4, 1, 24, 24)
    small.fields["pos"] *= (0.4, 0.1, 0.4)
    one = padded(small, 2049)
    o = OracleWorld(one)
    o.calculate_derived()
    with World(scenes.concat([one] * worlds), contact_capacity=200 * worlds) as w:
        for _ in range(2):
            w.integrate(one.dt)
            w.narrowphase()
            w.resolve(one.dt, 4)
            o.integrate(one.dt)
            cs = o.narrowphase()
            o.resolve(cs, one.dt, 4 * len(cs))
        assert len(cs) > 24 and (w.contact_counts() == len(cs)).all()
        it = w.resolver_iterations()
        assert (it == it[0]).all() and it[0].min() > 0
        for k, width in (("pos", 3), ("vel", 3), ("rot", 3), ("quat", 4)):
            got = w.get(k).reshape(worlds, -1)
            assert (got == got[0]).all(), k
            assert same(got[0], o.a[k][:width * o.n]), k
