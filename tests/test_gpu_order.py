"""The order in which worlds start (longest first, from the launch before)
changes no result: around the number of worlds from which it is computed and
the threads that compute it, every step's worlds equal the same worlds run
alone."""
import numpy as np
import pytest

from cubez_amd import World, scenes
from tests.test_gpu_parity import STATE, same

pytestmark = pytest.mark.gpu


def _part(sc, lo, hi):
    b0, b1 = int(sc.body_off[lo]), int(sc.body_off[hi])
    p0, p1 = int(sc.plane_off[lo]), int(sc.plane_off[hi])
    return scenes.Scene(sc.body_off[lo:hi + 1] - b0, sc.plane_off[lo:hi + 1] - p0, sc.plane_normal[p0:p1],
                        sc.plane_offset[p0:p1], {k: v[b0:b1] for k, v in sc.fields.items()}, name="part", dt=sc.dt), b0, b1


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("worlds", [256, 257, 1023, 1025])
def test_worlds_equal_themselves_in_a_small_batch(worlds, precision):
    sc = scenes.batched(2, worlds, 1, 40)
    with World(sc, precision=precision) as w:
        w.step(sc.dt, 110, 4)
        w.step(sc.dt, 3, 4)
        for lo in (0, worlds // 2, worlds - 30):
            part, b0, b1 = _part(sc, lo, lo + 30)
            with World(part, precision=precision) as v:
                v.step(sc.dt, 110, 4)
                v.step(sc.dt, 3, 4)
                for k in STATE:
                    assert same(w.get(k)[b0:b1], v.get(k)), (lo, k)
