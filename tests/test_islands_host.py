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


@pytest.fixture(scope="module")
def lib_o0(tmp_path_factory):
    return emu.build(str(tmp_path_factory.mktemp("emu_o0")), "-O0")


STATE = ("pos", "quat", "vel", "rot", "iit_world", "transform", "motion", "flags")
INTERNALS = ("pen", "cvel", "ddv", "c2w", "rel")


def _at_contacts(sc, at, world=0):
    o = OracleWorld(sc, world)
    o.calculate_derived()
    o.step(sc.dt, at, 4)
    o.integrate(sc.dt)
    return o, o.narrowphase()


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_no_access_past_the_workgroups_lds(lib_o0, precision):
    """Islands that leave lanes of their group without a contact, in every class
    of one contact per lane."""
    sc = _pile(200, 1.0)
    o, cs = _at_contacts(sc, 200)
    rc, _, iters, left = emu.resolve(lib_o0, o, cs, sc.dt, precision=precision)
    assert (rc, left) == (0, 0) and min(iters) > 0


def _check(lib, o, cs, dt, mult=4, fixed=0, flags=0, **kw):
    """The emulated resolve against the oracle's, which the world then takes."""
    rc, got, iters, left = emu.resolve(lib, o, cs, dt, mult, fixed, **kw)
    assert rc == 0, rc
    before = dict(o.counters())
    out = o.resolve(cs, dt, fixed or mult * len(cs), flags)
    after = o.counters()
    assert left == 0
    assert iters == (after["pos_iters"] - before["pos_iters"], after["vel_iters"] - before["vel_iters"])
    for k in STATE:
        assert np.array_equal(got[k].T.reshape(-1), o.a[k], equal_nan=True), k
    for k in INTERNALS:
        assert np.array_equal(got[k].T.reshape(-1), np.asarray(out[k]).reshape(-1), equal_nan=True), k


@pytest.mark.parametrize("across", [False, True])
def test_batches_are_dealt_out_once(lib, across):
    """Dozens of small islands of every class: each is run by exactly one wave,
    also when the waves draw their tickets lane by lane in turn."""
    sc = _pile(200, 1.0)
    o, cs = _at_contacts(sc, 200)
    _check(lib, o, cs, sc.dt, across=across)


def _bits(got):
    return {k: got[k] for k in (*STATE, *INTERNALS, "labels")}


@pytest.mark.parametrize("n,squeeze,at", [(64, 1.0, 300), (200, 1.0, 240), (200, 0.5, 200)])
def test_no_room_for_the_logs(lib, n, squeeze, at):
    """A world over its budget whose logs find no room runs as one island: the
    oracle's result, without the serial kernel."""
    sc = _pile(n, squeeze)
    o, cs = _at_contacts(sc, at)
    _check(lib, o, cs, sc.dt, mult=1, log_cap=10)


@pytest.mark.parametrize("kind", [emu.PLAIN, emu.LABEL, emu.MAT])
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("mult,fixed", [(1, 0), (2, 0), (4, 33)])
def test_merged_logs_equal_one_island(lib, kind, precision, mult, fixed):
    """Two ways to stop a world at its budget, the merged logs of its islands and
    one island of all of its contacts: the same bits in every kind, labels and
    iteration counts included."""
    sc = _pile(120, 0.4)
    o, cs = _at_contacts(sc, 200)
    rng = np.random.default_rng(3)
    cs["friction"] = rng.uniform(0.0, 1.0, len(cs))
    cs["friction"][::7] = 0.0
    cs["restitution"] = rng.uniform(0.0, 0.5, len(cs))
    a = emu.resolve(lib, o, cs, sc.dt, mult, fixed, precision, kind)
    b = emu.resolve(lib, o, cs, sc.dt, mult, fixed, precision, kind, log_cap=0)
    budget = fixed or mult * len(cs)
    assert a[0] == b[0] == 0 and a[3] == b[3] == 0 and a[2] == b[2] and budget in a[2]
    for k, v in _bits(a[1]).items():
        assert np.array_equal(v, b[1][k], equal_nan=True), k
    assert kind != emu.LABEL or np.abs(a[1]["labels"]).max() > 0


@pytest.mark.parametrize("threads", [256, 128])
@pytest.mark.parametrize("n,squeeze,at", [(12, 1.0, 60), (64, 1.0, 100), (200, 1.0, 120), (120, 0.4, 200)])
def test_stopped_at_the_budget(lib, n, squeeze, at, threads):
    """Budgets around every rule of a world that exceeds its own: one island of
    all contacts (small, or short), logs from the first iteration, logs and
    checkpoints of an island that runs for a quarter of the budget."""
    sc = _pile(n, squeeze)
    for i, budget in enumerate((1, 31, 96, 97, 128, 131, 200, 256, 399, 700, 1500)):
        o, cs = _at_contacts(sc, at)
        if len(cs):
            _check(lib, o, cs, sc.dt, fixed=budget, log_cap=0 if i % 4 == 3 else 200000, threads=threads)
