"""The IVF index lays its lists out once, and again whenever they can have changed."""
import numpy as np
from vector_store.ivf import IndexIVFFlat


def _index(lists):
    ivf = IndexIVFFlat.__new__(IndexIVFFlat)  # the lists alone, without a device
    ivf.nlist, ivf._lists, ivf._flat, ivf._lent = len(lists), lists, None, False
    return ivf


def test_layout_is_kept():
    ivf = _index([[0, 3], [], [1, 2]])
    ids, starts, sizes = ivf._flat_lists()
    assert ids.tolist() == [0, 3, 1, 2] and starts.tolist() == [0, 2, 2, 4]
    assert sizes.tolist() == [2, 0, 2]
    assert ivf._flat_lists()[0] is ids


def test_lists_changed_by_a_holder_are_seen():
    # a holder may move ids between two searches without asking for the lists again
    ivf = _index([[0, 3], [], [1, 2]])
    ivf._flat_lists()
    held = ivf.inv_lists
    ivf._flat_lists()
    held[1].append(held[0].pop())
    ids, starts, sizes = ivf._flat_lists()
    assert ids.tolist() == [0, 3, 1, 2] and starts.tolist() == [0, 1, 2, 4]
    assert np.array_equal(sizes, [1, 1, 2])
