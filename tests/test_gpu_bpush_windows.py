"""The beam push with its particles sorted into bins and the fields of a bin in LDS, against the push of one lane per particle
that gathers from F, bit for bit."""
import numpy as np
import pytest

import g3d_amd
from decks import bunch_deck

pytestmark = pytest.mark.gpu


# the shortest lists, and both sides of the length from which the particles are sorted by radix passes
@pytest.mark.parametrize("count", [1, 3, 5000, 131072, 131073])
def test_windowed_push_is_the_plain_push(count):
    a, b = g3d_amd.Sim(bunch_deck(nmacro=140000)), g3d_amd.Sim(bunch_deck(nmacro=140000))
    b.call("bpush_windows", 0)
    a.init(); b.init()
    p = a.array("parts")
    assert len(p) > 131073
    for s in (a, b):
        s.set_particles(p[:count])
        s.call("push", 0.0, 20.0)
    pa, pb = a.array("parts"), b.array("parts")
    assert len(pa) == count and not np.array_equal(pa["x"], p["x"][:count])
    for f in pa.dtype.names:
        np.testing.assert_array_equal(pa[f], pb[f], err_msg=f)
