"""The ordered beam deposit on the periodic grid against numpy's sequential sums (np.add.at adds in list order), bit for
bit, and the current spectra against numpy's transforms: bunches across the periodic edge, on tile corners, in one cell,
bins of one particle and of many chunks, the smallest grids of whole tiles and one without."""
import ctypes as C

import numpy as np
import pytest

import g3d_amd
from test_gpu_sponge_fused import tables

pytestmark = pytest.mark.gpu
D = g3d_amd.DevArray


def stencil(x, d, n):
    xi = x / d
    i0 = np.floor(xi + 0.5)
    f = xi - i0
    a, b = 0.5 - f, 0.5 + f
    return [(i0.astype(np.int64) + k - 1) % n for k in range(3)], [0.5 * a * a, 0.75 - f * f, 0.5 * b * b]


@pytest.mark.parametrize("nx,ny,ns,n,centre,sigma", [
    (16, 16, 4, 1, (8, 8), 0.0), (16, 32, 5, 255, (0, 0), 1.0), (32, 16, 3, 257, (8, 8), 0.3), (64, 64, 40, 5000, (31, 3), 6.0),
    (32, 32, 2, 20000, (16, 16), 1.6), (128, 64, 9, 30001, (100, 60), 40.0), (8, 16, 4, 700, (3, 3), 1.0),
    (4, 64, 4, 300, (2, 30), 3.0)])
def test_deposit_order_and_spectra(nx, ny, ns, n, centre, sigma):
    check(nx, ny, ns, n, centre, sigma)


# a bin of exactly 32 particles (the last that a wave takes), of 33, of 512 (the last of one chunk), of 513; particles all
# over a window (nearly all bins of few); the longest list whose keys are merged, and one particle more
@pytest.mark.parametrize("nx,ny,ns,n,centre,sigma", [
(16, 16, 2, 39, (8, 8), 0.0), (16, 16, 3, 67, (8, 8), 0.0), (16, 16, 2, 604, (8, 8), 0.0), (16, 16, 3, 1107, (8, 8), 0.0),
    (32, 64, 20, 6000, (16, 32), 30.0), (32, 32, 6, 32768, (16, 16), 3.0), (32, 32, 6, 32769, (16, 16), 3.0)])
def test_deposit_of_few_and_many(nx, ny, ns, n, centre, sigma):
    check(nx, ny, ns, n, centre, sigma)


def test_both_sorts_on_the_same_buffers():
    """the record sort (8 x 16 points) and the particle sort (32 x 32) in turn on the library's buffers, each call longer
    than the other sort's buffers and, in the records they share, no longer than what the call before left"""
    for nx, ny, n in ((8, 16, 40000), (32, 32, 100000), (8, 16, 120000), (32, 32, 300000)):
        check(nx, ny, 4, n, (nx // 2, ny // 2), 2.0)


def check(nx, ny, ns, n, centre, sigma):
    r = np.random.default_rng(n)
    dx, dy, h = 0.9, 0.7, 0.25
    p = np.zeros(n, dtype=g3d_amd.PARTICLE)
    p["x"] = dx * (centre[0] + sigma * r.standard_normal(n)); p["y"] = dy * (centre[1] + sigma * r.standard_normal(n))
    p["zeta"] = h * (ns - 1) * r.uniform(-0.05, 1.05, n)
    p["px"], p["py"] = r.standard_normal((2, n))
    p["pz"] = 5 + r.standard_normal(n)
    p["w"] = r.uniform(0.5, 1.5, n); p["q"] = -1; p["alive"] = 1
    p["alive"][::17] = 0
    p["px"][:2] = 0
    (kx, kxs, fx), (ky, kys, fy) = tables(nx, dx), tables(ny, dy)
    d = {k: D(v) for k, v in (("kx", kx), ("kxs", kxs), ("fx", fx), ("ky", ky), ("kys", kys), ("fy", fy),
                              ("hcg", np.full(ns + 3, h)), ("half", np.full(ns, 0.5)), ("ia", np.full(ny, 1 / dy)))}
    a = lambda k: d[k].ptr.value
    nk = nx * ny
    plan = g3d_amd.FftPlan(nx, ny)
    spec = g3d_amd.SpecCtx(nx=nx, ny=ny, ns=ns, N=ns, a=0, nk=nk, kx=a("kx"), ky=a("ky"), kxs=a("kxs"), kys=a("kys"),
                           filt=a("fx"), filty=a("fy"), hcg=a("hcg"), wlo=a("half"), whi=a("half"), a2=0.0, keep0=1,
                           plan=plan.h.value)
    zax = g3d_amd.Axis(X=None, n=ns, uniform=1, x0=0.0, ih=1 / h)
    jw, scr = D(nbytes=3 * (ns + 3) * nk * 8), D(nbytes=(ns + 1) * nk * 16)
    jk = [D(nbytes=(ns + 1) * nk * 16) for _ in range(3)]
    parts = g3d_amd.DeviceParts(p)
    for _ in range(2):                     # the second call on the library's buffers of the first
        g3d_amd.kernel_call("g3d_bunch_currents", C.byref(spec), C.byref(zax), d["ia"].ptr, d["ia"].ptr, dx, dy, 1, 1,
                            C.byref(parts.c), n, jw.ptr, jk[0].ptr, jk[1].ptr, jk[2].ptr, scr.ptr)
    m = np.floor(p["zeta"] * (1 / h)).astype(np.int64)
    s = p[(p["alive"] == 1) & (m >= 0) & (m <= ns - 2)]
    hw = np.floor(s["zeta"] * (1 / h)).astype(np.int64) + 2
    g = np.sqrt(1 + s["px"] * s["px"] + s["py"] * s["py"] + s["pz"] * s["pz"])
    vx, vy, vz = s["px"] / g, s["py"] / g, s["pz"] / g
    f = s["q"] * s["w"] / (h * dx)
    ix, wx = stencil(s["x"], dx, nx)
    jy, wy = stencil(s["y"], dy, ny)
    want = np.zeros((3, (ns + 3) * nk))
    cells, vals = [], []
    for v in range(3):
        for u in range(3):
            w = f * wx[u] * wy[v] * (1 / dy)
            cells.append(hw * nk + jy[v] * nx + ix[u])
            vals.append([w * vx / vz, w * vy / vz, w])
    cells, vals = np.array(cells).T.reshape(-1), np.array(vals)       # particle by particle
    for k in range(3):
        np.add.at(want[k], cells, vals[:, k].T.reshape(-1))
    assert np.array_equal(jw.get(np.float64).reshape(3, -1), want)
    J = want.reshape(3, ns + 3, ny, nx)
    v = 0.25 * J[:, :ns + 1] + 0.5 * J[:, 1:ns + 2] + 0.25 * J[:, 2:ns + 3]
    v[:, 0] = v[:, ns] = 0
    spectra = fx[None, None, None, :] * fy[None, None, :, None] * np.fft.fft2(v)
    # 2 log2(nx ny) butterflies of rounding 1.1e-16 each, on planes of one scale
    scale = np.linalg.norm(spectra)
    for k in range(3):
        got = jk[k].get(np.complex128).reshape(ns + 1, ny, nx)
        assert np.linalg.norm(got - spectra[k]) <= 1e-14 * scale
