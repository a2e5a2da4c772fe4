"""The sponge and the real fields with their steps fused into the transforms, against the same formulas in 64 bits
(numpy), on the smallest and the most lopsided planes; and column-major against row-major modes in the engine."""
import ctypes as C

import numpy as np
import pytest

import g3d_amd
from decks import group_rel_l2, plasma_deck

pytestmark = pytest.mark.gpu
D = g3d_amd.DevArray


def tables(n, d):
    m = np.arange(n)
    ks = 2 * np.pi * np.where(m <= n // 2, m, m - n) / (n * d)
    k = ks.copy()
    k[n // 2] = 0
    f = np.cos(0.5 * ks * d) ** 2
    f[n // 2] = 0
    return k, ks, f


@pytest.mark.parametrize("sponge", [0, 1])
@pytest.mark.parametrize("nx,ny,ns", [(2, 2, 1), (2, 16, 3), (16, 2, 4), (8, 1024, 3), (1024, 8, 2), (64, 32, 33), (256, 128, 5)])
def test_sponge_and_real_fields(nx, ny, ns, sponge):
    r = np.random.default_rng(nx + ny)
    dx, dy, h, beta, gm2 = 0.9, 0.7, 0.25, 0.99, 1 - 0.99 ** 2
    (kx, kxs, fx), (ky, kys, fy) = tables(nx, dx), tables(ny, dy)
    hcg, half = np.full(ns + 3, h), np.full(ns, 0.5)
    a = {n: np.fft.fft2(r.standard_normal((ns + (n == "jkz"), ny, nx))) for n in
         ("Rx", "Ry", "Lx", "Ly", "Ez", "Bz", "jkz")}
    mx, my = r.uniform(0.8, 1, nx), r.uniform(0.8, 1, ny)
    d = {n: D(v) for n, v in (("kx", kx), ("kxs", kxs), ("fx", fx), ("ky", ky), ("kys", kys), ("fy", fy), ("hcg", hcg),
                              ("half", half), ("mx", mx), ("my", my))}
    plan = g3d_amd.FftPlan(nx, ny)
    p = lambda n: d[n].ptr.value
    spec = g3d_amd.SpecCtx(nx=nx, ny=ny, ns=ns, N=ns, a=0, nk=nx * ny, kx=p("kx"), ky=p("ky"), kxs=p("kxs"), kys=p("kys"),
                           filt=p("fx"), filty=p("fy"), hcg=p("hcg"), wlo=p("half"), whi=p("half"), a2=0.0, keep0=1,
                           plan=plan.h.value)
    arr = {n: D(v.reshape(-1)) for n, v in a.items()}
    F = D(nbytes=6 * (ns + 2) * nx * ny * 4)
    scr = D(nbytes=5 * ns * nx * ny * 16)
    g3d_amd.kernel_call("g3d_sponge_real_fields", C.byref(spec), sponge, d["mx"].ptr, d["my"].ptr, beta, gm2,
                        *[arr[n].ptr for n in ("Rx", "Ry", "Lx", "Ly", "Ez", "Bz", "jkz")], F.ptr, scr.ptr)
    Rx, Ry = a["Rx"], a["Ry"]
    bx = by = np.zeros(1)
    if sponge:
        KX, KY = kx[None, None, :], ky[None, :, None]
        k2 = KX ** 2 + KY ** 2
        ik2 = np.where(k2 > 0, 1 / np.where(k2 > 0, k2, 1), 0)
        rho = np.zeros((ns + 2, ny, nx), complex)
        rho[1:-1] = 0.5 * (a["jkz"][:-1] + a["jkz"][1:])
        psi = (rho[1:-1] + gm2 * (rho[2:] - 2 * rho[1:-1] + rho[:-2]) / (h * h) * ik2) * ik2
        bx, by = -(1 + beta) * 1j * KX * psi, -(1 + beta) * 1j * KY * psi
        z = np.fft.fft2(mx[None, None, :] * my[None, :, None] * np.fft.ifft2((Rx - bx) + 1j * (Ry - by)))
        zm = np.conj(np.roll(z[:, ::-1, ::-1], (1, 1), (1, 2)))
        Rx, Ry = 0.5 * (z + zm) + bx, -0.5j * (z - zm) + by
    # 4 log2(nx ny) butterflies of rounding 1.1e-16 each way, relative to the plane that is transformed: R_x + i R_y less
    # the bound field (which 1/k^4 makes the larger on a long box), added back afterwards
    scale = sum(np.linalg.norm(v) for v in (Rx, Ry, bx, by))
    for n, want in (("Rx", Rx), ("Ry", Ry)):
        got = arr[n].get(np.complex128).reshape(want.shape)
        assert np.linalg.norm(got - want) <= 1e-13 * scale, n
    R, L, Z = [np.fft.ifft2(u + 1j * v) for u, v in ((Rx, Ry), (a["Lx"], a["Ly"]), (a["Ez"], a["Bz"]))]
    want = np.stack([0.5 * (R.real + L.real), 0.5 * (R.imag + L.imag), Z.real, 0.5 * (L.imag - R.imag),
                     0.5 * (R.real - L.real), Z.imag])
    got = F.get(np.float32).reshape(6, ns + 2, ny, nx)
    assert not got[:, ns:].any()
    assert np.abs(got[:, :ns] - want).max() <= 1.2e-7 * np.abs(want).max()


@pytest.mark.parametrize("nx,ny", [(32, 64), (64, 32)])
def test_column_major_modes_give_the_same_fields(monkeypatch, nx, ny):
    """one step of the plasma deck with the modes column-major (the default) and row-major: R, L, E_z, B_z per slice to the
    FP64 parity bar"""
    out = {}
    for cm in ("0", "1"):
        monkeypatch.setenv("G3D_PASS_CM", cm)
        sim = g3d_amd.Sim(plasma_deck(nx=nx, ny=ny, nz=33))
        sim.init()
        sim.step()
        out[cm] = [sim.array(n) for n in ("Rx", "Ry", "Lx", "Ly", "Ez", "Bz")], sim.array("F")
        sim.close()
    assert group_rel_l2(out["1"][0], out["0"][0], 33) <= 1e-12
    assert np.abs(out["1"][1] - out["0"][1]).max() <= 1.2e-7 * np.abs(out["0"][1]).max()
