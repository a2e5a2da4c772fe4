"""The kernel-level C ABI (include/g3d.h) against outputs of the reference's CPU build that are kept in tests/golden, and,
where those hold none, against the same formulas in numpy: what test_gpu_kabi.py compares with that build itself, where it
is absent."""
import ctypes as C
import os

import numpy as np
import pytest

import g3d_amd
import golden_inputs as gi
from test_gpu_kabi import Tables

pytestmark = pytest.mark.gpu
D = g3d_amd.DevArray
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
STATE = ("x", "y", "zeta", "px", "py", "pz", "z", "alive")


def gold(name):
    return np.load(os.path.join(GOLD, name + ".npz"))


def test_stream_halfcell():
    g = gold("stream_pass")
    deck = gi.small_deck()
    t = Tables(g3d_amd.Sim(deck))
    F, J, parts = D(g["F"]), D(nbytes=g["jsr"].nbytes), g3d_amd.DeviceParts(g["parts_in"])
    pc = t.push(deck, F, 5.0)
    pc.X0, pc.Y0 = float(g["X0"]), float(g["Y0"])
    sc = g3d_amd.StreamCtx(pc=pc, zs=t.d["zs"].ptr.value, J=J.ptr.value, ia=t.d["iA"].ptr.value, id=t.d["iD"].ptr.value,
                           Delta=5.0, s1=5.0, sTrap=5.0 + (deck.c.trap_advance - 1) * 5.0, vz_beam=deck.c.vz_beam,
                           n=gi.STREAM_N)
    g3d_amd.kernel_call("g3d_stream_halfcell", C.byref(sc), C.byref(parts.c), C.byref(parts.c), parts.n)
    got = parts.records()
    for f in STATE:
        assert np.array_equal(got[f], g["parts_out"][f]), f
    # the sums of some ten terms in another order
    assert np.abs(J.get(np.float64) - g["jsr"]).max() <= 1e-13 * np.abs(g["jsr"]).max()


def test_stream_spectra():
    g = gold("stream_spectra")
    deck = gi.small_deck(smooth=float(g["a2"]) ** 0.5)
    t = Tables(g3d_amd.Sim(deck))
    plan = g3d_amd.FftPlan(8, 8)
    J, jsn, scr = D(g["J"]), D(nbytes=g["jsn"].nbytes), D(nbytes=6 * 64 * 16)
    g3d_amd.kernel_call("g3d_stream_spectra", C.byref(t.spec(deck, plan, keep0=deck.c.box_mean)), J.ptr, jsn.ptr, scr.ptr)
    assert np.abs(jsn.get(np.complex128) - g["jsn"]).max() <= 1e-14 * np.abs(g["jsn"]).max()


def test_bunch_push():
    g = gold("push")
    deck = gi.bunch_small_deck()
    sim = g3d_amd.Sim(deck)
    sim.init()
    t = Tables(sim)
    F, parts = D(g["F"]), g3d_amd.DeviceParts(g["parts_in"])
    pc = t.push(deck, F, 20.0)
    pc.X0, pc.Y0 = float(g["X0"]), float(g["Y0"])
    L = sim.array("laser")
    pc.laser = g3d_amd.PlaneWave(int(L[0]), int(L[1]), *L[2:])
    g3d_amd.kernel_call("g3d_bunch_push", C.byref(pc), C.byref(parts.c), 0, parts.n, 0.0)
    got = parts.records()
    for f in STATE:          # the wave calls exp, cos and sin, whose last bits are the library's
        assert np.allclose(got[f], g["parts_out"][f], rtol=1e-13, atol=0), f


def test_bunch_currents():
    g = gold("bunch_deposit")
    deck = gi.bunch_small_deck()
    t = Tables(g3d_amd.Sim(deck))
    i, plan, parts = t.info, g3d_amd.FftPlan(8, 8), g3d_amd.DeviceParts(g["parts"])
    jw, scr = D(nbytes=g["jw"].nbytes), D(nbytes=(i["ns"] + 1) * i["nk"] * 16)
    jk = [D(nbytes=(i["ns"] + 1) * i["nk"] * 16) for _ in range(3)]
    zax = t.zax(deck)
    g3d_amd.kernel_call("g3d_bunch_currents", C.byref(t.spec(deck, plan)), C.byref(zax), t.d["iA"].ptr, t.d["iD"].ptr,
                        i["dx"], i["dy"], deck.c.zeta_filter, 1, C.byref(parts.c), parts.n, jw.ptr, jk[0].ptr, jk[1].ptr,
                        jk[2].ptr, scr.ptr)
    assert np.array_equal(jw.get(np.float64), g["jw"])


def grid(nx=16, ny=8, nz=24):
    d = g3d_amd.Deck(gi.LAMBDA0).grid(nx, ny, nz, 20.0, 9.0, 0.4 * (nz - 1))
    d.set(dz=5.0, move_x=0, move_y=0)
    t = Tables(g3d_amd.Sim(d))
    h = {k: t.sim.array(k) for k in ("kx", "ky", "kxs", "kys", "hcg", "wlo", "whi")}
    return d, t, h, g3d_amd.FftPlan(nx, ny)


def test_comoving():
    """-(gm2 d^2/dzeta^2 - k^2) psi = rho / beta per mode as a dense real system, R = -(1 + beta) i k psi"""
    d, t, h, plan = grid()
    N, nx, ny, nk = t.info["N"], d.c.nx, d.c.ny, t.info["nk"]
    r = np.random.default_rng(3)
    beta = 0.98
    gm2 = 1 - beta * beta
    jkz = np.fft.fft2(r.standard_normal((N + 1, ny, nx))).reshape(N + 1, nk)
    dj, outs, scr = D(jkz.reshape(-1)), [D(np.full(N * nk, 7.0 + 1j)) for _ in range(4)], D(nbytes=2 * N * nk * 16)
    g3d_amd.kernel_call("g3d_comoving", C.byref(t.spec(d, plan)), dj.ptr, beta, gm2, *[o.ptr for o in outs], scr.ptr)
    hm, hp = h["hcg"][1:N + 1], h["hcg"][2:N + 2]
    k2 = (h["kx"][None, :] ** 2 + h["ky"][:, None] ** 2).reshape(-1)
    A = np.zeros((nk, N, N))
    j = np.arange(N)
    A[:, j, j] = k2[:, None] + gm2 * 2 / (hm * hp)
    A[:, j[1:], j[:-1]] = -gm2 * 2 / ((hm + hp) * hm)[1:]
    A[:, j[:-1], j[1:]] = -gm2 * 2 / ((hm + hp) * hp)[:-1]
    rho = (h["wlo"][:N, None] * jkz[:-1] + h["whi"][:N, None] * jkz[1:]) / beta
    psi = np.linalg.solve(A, rho.T[:, :, None])[:, :, 0].T
    kx, ky = np.tile(h["kx"], ny), np.repeat(h["ky"], nx)
    # two solvers of the same system: roundings times its condition, k2 + 4 gm2 / h^2 over k2 + gm2 (pi / L)^2 (about
    # 10^4 on this grid at k = 0, whose R is zero; some 20 at the smallest other k)
    for got, k in zip(outs, (kx, ky)):
        want = -(1 + beta) * 1j * k[None, :] * psi
        assert np.linalg.norm(got.get(np.complex128) - want.reshape(-1)) <= 1e-13 * np.linalg.norm(want)
    assert not outs[2].get(np.complex128).any() and not outs[3].get(np.complex128).any()


@pytest.mark.parametrize("nxs,nys", [(3, -2), (-5, 0), (16, 8)])
def test_window_shift_and_centroid(nxs, nys):
    d, t, h, plan = grid()
    ns, nx, ny, nk, dx, dy = t.info["ns"], d.c.nx, d.c.ny, t.info["nk"], t.info["dx"], t.info["dy"]
    r = np.random.default_rng(5)
    a = [r.standard_normal((n, nk)) + 1j * r.standard_normal((n, nk)) for n in (ns, ns + 1)]
    F = r.standard_normal((6, ns + 2, ny, nx)).astype(np.float32)
    p = np.zeros(1000, dtype=g3d_amd.PARTICLE)
    p["x"], p["y"], p["w"] = r.uniform(0, 20, 1000), r.uniform(0, 9, 1000), r.uniform(0.5, 1.5, 1000)
    p["alive"] = 1
    p["alive"][::9] = 0
    p["sp"][::7] = 1
    parts, dF, dFs, da = g3d_amd.DeviceParts(p), D(F.reshape(-1)), D(nbytes=F.nbytes), [D(v.reshape(-1)) for v in a]
    out = np.zeros(3)
    g3d_amd.kernel_call("g3d_bunch_centroid", C.byref(parts.c), 1000, 0.25, -0.5, out.ctypes.data_as(C.c_void_p))
    q = p[(p["alive"] == 1) & (p["sp"] <= 0)]
    np.testing.assert_allclose(out, [(q["w"] * (q["x"] + 0.25)).sum(), (q["w"] * (q["y"] - 0.5)).sum(), q["w"].sum()], rtol=1e-12)
    counts = (C.c_long * 2)(ns, ns + 1)
    ptrs = (C.c_void_p * 2)(*[v.ptr.value for v in da])
    g3d_amd.kernel_call("g3d_window_shift", C.byref(t.spec(d, plan)), nxs, nys, dx, dy, ptrs, counts, 2, dF.ptr, dFs.ptr,
                        C.byref(parts.c), 1000)
    ph = h["kxs"][None, :] * (nxs * dx) + h["kys"][:, None] * (nys * dy)
    for got, v in zip(da, a):            # a product of numbers of one size: a few roundings and those of sin and cos
        np.testing.assert_allclose(got.get(np.complex128).reshape(v.shape), v * np.exp(1j * ph).reshape(-1), rtol=0, atol=1e-14 * np.abs(v).max())
    assert np.array_equal(dF.get(np.float32).reshape(F.shape), np.roll(F, (-nys, -nxs), (2, 3)))
    got = parts.records()
    assert np.array_equal(got["x"], p["x"] - nxs * dx) and np.array_equal(got["y"], p["y"] - nys * dy)


def test_real_fields_slice():
    d, t, h, plan = grid()
    ns, nx, ny, nk = t.info["ns"], d.c.nx, d.c.ny, t.info["nk"]
    r = np.random.default_rng(7)
    a = [np.fft.fft2(r.standard_normal((ny, nx))) for _ in range(6)]
    F, scr, da = D(nbytes=6 * (ns + 2) * nk * 4), D(nbytes=3 * nk * 16), [D(v.reshape(-1)) for v in a]
    n = 5
    g3d_amd.kernel_call("g3d_real_fields_slice", C.byref(t.spec(d, plan)), *[v.ptr for v in da], C.c_void_p(F.ptr.value + n * nk * 4),
                        (ns + 2) * nk, scr.ptr)
    Rx, Ry, Lx, Ly, Ez, Bz = [np.fft.ifft2(v).real for v in a]
    want = np.stack([0.5 * (Rx + Lx), 0.5 * (Ry + Ly), Ez, 0.5 * (Ly - Ry), 0.5 * (Rx - Lx), Bz])
    got = F.get(np.float32).reshape(6, ns + 2, ny, nx)
    assert np.abs(got[:, n] - want).max() <= 1.2e-7 * np.abs(want).max()
    got[:, n] = 0
    assert not got.any()
