"""The broadphase's sweep and sort at the edges of their tiles: 64 positions
and 128 boxes per step of the sweep, its 2048 collected overlaps; the sort's
tiles of 1024 keys up to 131072 keys and of 4096 above, the scan of their
histograms from more than 128 tiles (524288 keys) on."""
import numpy as np
import pytest

from cubez_amd import World, scenes
from tests.test_gpu_broadphase import _compare
from tests.test_gpu_sort import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("squeeze", [1.0, 0.12])
def test_sweep_on_worlds_around_its_tiles(squeeze):
    """Worlds of 1 to 257 bodies side by side in the sorted order, spread out
    and squeezed until one workgroup meets far more than 2048 overlaps (257
    bodies within 8 m, boxes of 3 to 9 m)."""
    sizes = [1, 2, 63, 64, 65, 127, 128, 129, 191, 192, 193, 257]
    base = scenes.batched(8, 1, sum(sizes), sum(sizes))
    f = dict(base.fields)
    f["pos"] = f["pos"].copy()
    for k, n in enumerate(sizes):
        a = sum(sizes[:k])
        f["pos"][a:a + n, 0] *= squeeze * np.sqrt(n / sum(sizes))
        f["pos"][a:a + n, 2] *= squeeze * np.sqrt(n / sum(sizes))
    nw = len(sizes)
    sc = scenes.Scene(np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32), np.arange(nw + 1, dtype=np.int32),
                      np.tile([0.0, 1.0, 0.0], (nw, 1)), np.zeros(nw), f, name="edges", dt=base.dt)
    with World(sc, contact_capacity=400_000) as w:
        w.calculate_derived()
        total, checked = _compare(w)
        if squeeze < 1.0:  # the largest world alone: most of its pairs overlap
            assert checked > 257 * 256 // 2
        w.step(sc.dt, 3, 4)
        _compare(w)


def test_sort_around_its_tiles_and_scan():
    rng = np.random.default_rng(3)
    with World() as w:
        for n in (255, 257, 1023, 1024, 1025, 130_048, 131_071, 131_072, 131_073, 524_287, 524_288, 524_289, 700_001):
            _check(w, rng.integers(0, 2**63, n, dtype=np.int64).astype(np.uint64) >> np.uint64(rng.integers(0, 40)))
            _check(w, rng.integers(0, 3, n).astype(np.uint64), with_vals=False)
