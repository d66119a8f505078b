"""What a narrowphase that finds no room reports."""
import ctypes

import numpy as np
import pytest

from cubez_amd import World, scenes

pytestmark = pytest.mark.gpu


def test_a_list_without_contact_slots_names_the_contacts():
    """5900 cubes in one place: more candidate pairs than the all-pairs
    narrowphase has slots for.  What it counted says nothing about the list of
    the call after it."""
    sc = scenes.batched(0, 1, 5900, 5900)
    sc.fields["pos"][:] = (0.0, -1.0, 0.0)
    with World(sc, contact_capacity=100) as w:
        w.calculate_derived()
        with pytest.raises(RuntimeError, match="candidate list exceeded"):
            w.narrowphase()
        one = np.arange(200, dtype=np.int32)
        with pytest.raises(RuntimeError, match="contact capacity exceeded"):
            w.narrowphase_pairs(one, np.full(200, -1, np.int32))


def test_a_failed_narrowphase_leaves_the_total_alone():
    sc = scenes.batched(0, 1, 64, 64)
    sc.fields["pos"][:, 1] = -1.0
    with World(sc, contact_capacity=100) as w:
        w.calculate_derived()
        total = ctypes.c_int64(-7)
        body, plane = np.arange(64, dtype=np.int32), np.full(64, -1, np.int32)
        for call in (lambda: w._lib.cbz_narrowphase(w._h, ctypes.byref(total)),
                     lambda: w._lib.cbz_narrowphase_pairs(w._h, 64, body.ctypes.data, plane.ctypes.data,
                                                          ctypes.byref(total)),
                     lambda: w._lib.cbz_narrowphase_broad(w._h, ctypes.byref(total), None)):
            assert call() != 0 and total.value == -7
