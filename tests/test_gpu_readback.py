"""Sim.array of large arrays (copied through pinned buffers by several threads) against what was written."""
import threading

import numpy as np
import pytest

import g3d_amd
import golden_inputs as gi

pytestmark = pytest.mark.gpu


# F of 64 x 64 points: the last size of the plain copy, the first of the staged one (a few chunks more than the buffers'),
# a long one with a short last chunk
@pytest.mark.parametrize("nz", [509, 510, 1501])
def test_large_array_round_trip(nz):
    d = g3d_amd.Deck(gi.LAMBDA0).grid(64, 64, nz, 64.0, 64.0, (nz - 1) * 0.5)
    d.set(dz=5.0, z_end=100.0, plasma_on=0)
    sim = g3d_amd.Sim(d)
    want = np.random.default_rng(nz).standard_normal(6 * (nz + 2) * 64 * 64).astype(np.float32)
    sim.set("F", want)
    got = [None, None]

    def read(k):
        got[k] = sim.array("F")
    threads = [threading.Thread(target=read, args=(k,)) for k in (0, 1)]      # the buffers belong to a call
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        assert np.array_equal(g.view(np.uint32), want.view(np.uint32))
