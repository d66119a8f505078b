"""The island resolver's code on the CPU (tests/emu) against the oracle, bit
for bit."""
import numpy as np
import pytest

from cubez_amd import scenes
from oracle.cbz_oracle import OracleWorld
from tests import emu
from tests.test_gpu_islands import _pile


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return emu.build(str(tmp_path_factory.mktemp("emu")))


STATE = ("pos", "quat", "vel", "rot", "iit_world", "transform", "motion", "flags")
INTERNALS = ("pen", "cvel", "ddv", "c2w", "rel")


def _at_contacts(sc, at, world=0):
    o = OracleWorld(sc, world)
    o.calculate_derived()
    o.step(sc.dt, at, 4)
    o.integrate(sc.dt)
    return o, o.narrowphase()


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_no_access_past_the_workgroups_lds(lib, precision):
    """Islands that leave lanes of their group without a contact, in every class
    of one contact per lane."""
    sc = _pile(200, 1.0)
    o, cs = _at_contacts(sc, 200)
    rc, _, iters, left = emu.resolve(lib, o, cs, sc.dt, precision=precision)
    assert (rc, left) == (0, 0) and min(iters) > 0
