"""What the Python binding hands to the library for switches that take any
truth value."""
import numpy as np
import pytest

from lustrine_amd import gpu as G


class _Calls:
    def __init__(self):
        self.got = []

    def lus_pbf_set_build(self, handle, staged):
        self.got.append(staged)
        return 0


@pytest.mark.parametrize("given,want", [(True, 1), (False, 0), (1, 1), (0, 0), (2, 2), (2.0, 2), (None, 0), ("yes", 1), ("", 0),
                                        (0.5, 1), (7, 1), (-1, 1), (np.bool_(True), 1), (np.int64(2), 2), ([], 0)])
def test_build_switch(given, want):
    g = G.Gpu.__new__(G.Gpu)
    g._lib, g._h = _Calls(), None
    g.pbf_set_build(given)
    assert g._lib.got == [want]
    g._lib = None
