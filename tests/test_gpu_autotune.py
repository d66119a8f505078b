"""The autotuner of the resolver split, none of whose candidates differ: one is
timed for all, the first is set, the body state is as it was."""
import numpy as np
import pytest

from cubez_amd import World, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("surrogate", [False, True])
def test_one_candidate_is_timed_for_all(surrogate):
    from cubez_amd import surrogate as model
    sc = scenes.batched(2, 6, 8, 24)
    with World(sc, precision="f32") as w:
        if surrogate:
            model.install(w)
        w.step(sc.dt, 100, 4)
        before = w.checkpoint()
        r = w.autotune_resolver(sc.dt, 4, 3, ((7, 2), (0, 0), (257, 16)), surrogate=surrogate)
        assert r["split"] == (7, 2) == w.resolver_split()
        ms = list(r["ms_per_step"].values())
        assert len(ms) == 3 and ms[0] > 0 and ms == [ms[0]] * 3
        after = w.checkpoint()
        for k in ("pos", "vel", "rot", "quat", "motion", "flags"):
            x = w.get(k)
            w.restore(before)
            assert np.array_equal(x, w.get(k)), k
            w.restore(after)
        with pytest.raises(RuntimeError, match="negative split"):
            w.autotune_resolver(sc.dt, 4, 3, ((7, 2), (-1, 0)))
        assert w.resolver_split() == (7, 2)
