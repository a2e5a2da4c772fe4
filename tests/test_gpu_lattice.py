"""The fresh plasma made on the device against the host loader (the reference's order and values,
src/sim_plasma.cpp:43-90), and the ion statistics summed on the device against the list itself."""
import numpy as np
import pytest

import g3d_amd
from decks import LAMBDA0

pytestmark = pytest.mark.gpu
AMU = 1822.888486


def deck(yf, nx, ny, ppc, species, electrons=1, parabolic=0, a0=0.0, extra=None):
    d = g3d_amd.Deck(LAMBDA0)
    d.c.nx = nx; d.c.Lx = 40.0
    if yf:
        d.y_uniform(ny, 30.0)
    else:
        d.y_nodes(np.cumsum(0.3 + 0.1 * np.abs(np.arange(ny + 1) - ny // 2)) - 3.0)
    d.zeta_uniform(13, 12 * 0.5)
    d.set(dz=5.0, z_end=1000.0, plasma_on=1, n0=1e-2, ppc_x=ppc[0], ppc_y=ppc[1], move_x=0, sponge=4.0, sponge_y=4.0,
          free_electrons=electrons, parabolic=parabolic, channel_depth=0.3, r_channel=5.0)
    if yf:
        d.set(move_y=0)
    if "H" in species:
        d.add_ion(1.00794 * AMU, 1, 1, atoms=0.7, mobile=True, ionization=False)
    if "N" in species:
        d.add_ion(14.0067 * AMU, 0, 7, atoms=0.01, mobile=True, ionization=True,
                  ip_eV=(14.53413, 29.60125, 47.4453, 77.4735, 97.8901, 552.06732, 667.0461))
    if a0:
        d.add_grid_laser(a0=a0, waist=8.0, tau=2.0, zeta_c=3.0)
    return d


# tiles of 16 x 8 cells; ny not a multiple of 8 (the last row of tiles short), a row of tiles that holds only a wall
CASES = [(1, 32, 16, (2, 2), "", 1, 0), (1, 64, 32, (3, 1), "HN", 1, 1), (1, 32, 32, (2, 1), "N", 0, 0),
         (0, 32, 18, (2, 1), "HN", 1, 0), (0, 64, 25, (1, 3), "N", 1, 1), (0, 32, 17, (2, 2), "H", 0, 0)]


@pytest.mark.parametrize("yf,nx,ny,ppc,species,electrons,parabolic", CASES)
def test_device_lattice_is_the_host_list(monkeypatch, yf, nx, ny, ppc, species, electrons, parabolic):
    lists = []
    for host in ("0", "1"):
        monkeypatch.setenv("G3D_HOST_LATTICE", host)
        sim = g3d_amd.Sim(deck(yf, nx, ny, ppc, species, electrons, parabolic))
        sim.init()
        sim.call("load_plasma", 0.0, 5.0)
        lists.append((sim.array("strm"), sim.info()["born_cap"]))
        sim.close()
    assert len(lists[0][0]) == len(lists[1][0]) > 0 and lists[0][1] == lists[1][1]
    assert np.array_equal(lists[0][0], lists[1][0])


@pytest.mark.parametrize("yf,ny", [(1, 32), (0, 26)])
def test_ion_statistics_are_the_sums_of_the_list(yf, ny):
    """nitrogen freed by the laser: the weights per charge state and the freed charge (sums of at most 2^13 positive
    terms in another order: 1e-12 relative)"""
    sim = g3d_amd.Sim(deck(yf, 32, ny, (2, 1), "HN", a0=1.0))
    sim.init()
    sim.step()
    p, h = sim.array("strm"), sim.array("ion_stats1")
    n = p[p["sp"] == 4]
    Z = np.rint(n["q"]).astype(int)
    want = [n["w"][(Z == z) & (n["alive"] == 1)].sum() for z in range(8)] + [(Z * n["w"]).sum()]
    assert want[8] > 0
    np.testing.assert_allclose(h, want, rtol=1e-12)


def test_ion_statistics_of_a_species_without_ions_are_empty():
    """a step outside the plasma with one electron waiting to join the stream: the list holds no ion, and the statistics of
    an ionizing species are empty, not zeros"""
    d = deck(1, 32, 32, (2, 1), "HN")
    d.c.n_pz = 2
    d.c.pz_points[0], d.c.pz_points[1] = 0.0, 100.0
    d.c.pz_values[0], d.c.pz_values[1] = 0.0, 0.0
    sim = g3d_amd.Sim(d)
    sim.init()
    p = np.zeros(1, dtype=g3d_amd.PARTICLE)
    p["x"], p["y"], p["zeta"], p["z"] = 20.0, 15.0, 2.7, 0.0
    p["w"], p["q"], p["qm"], p["alive"], p["sp"] = 1e-3, -1, -1, 1, 1
    sim.set_joining(p)
    sim.step()
    assert sim.info()["nstrm"] == 1
    assert len(sim.array("ion_stats0")) == 0 and len(sim.array("ion_stats1")) == 0
