"""g3d_stream_halfcell on lists long enough to be streamed through tiles, and on shorter ones in the order of a lattice
(whose workgroups sum their deposits in a box), against the same particles streamed in short lists in no order (one
atomic per deposit)."""
import ctypes as C

import numpy as np
import pytest

import g3d_amd

pytestmark = pytest.mark.gpu
D = g3d_amd.DevArray
SHORT = 8000              # well below the length from which a list is tiled


def context(nx, ny, dx, dy, F, J, zs, ia, n, ns, s0, s1):
    h = zs[1] - zs[0]
    zax = g3d_amd.Axis(X=None, n=len(zs), uniform=1, x0=0.0, ih=1 / h)
    yax = g3d_amd.Axis(X=None, n=ny + 1, uniform=1, x0=0.0, ih=1 / dy)
    pc = g3d_amd.PushCtx(F=F.ptr.value, a=0, ns=ns, N=ns, nx=nx, ny=ny, self=1, yf=1, nk=nx * ny, dx=dx, dy=dy,
                         Lx=nx * dx, Ly=ny * dy, zax=zax, yax=yax, X0=0.0, Y0=0.0, zc=0.0, dz_push=s1 - s0,
                         push_phase=0.05, zhand=-1e300, zmax=zs[-1], ylo=-1e300, yhi=1e300, s1=s1, vz_min=0.0, hmin=h)
    z = D(np.asarray(zs))
    i = D(ia)
    sc = g3d_amd.StreamCtx(pc=pc, zs=z.ptr.value, J=J.ptr.value, ia=i.ptr.value, id=i.ptr.value, Delta=s1 - s0, s1=s1,
                           sTrap=s1, vz_beam=0.9, n=n)
    return sc, (z, i)


# the tiles' shapes: 16 x 8 (512 x 64 cells are 256 of them), 8 x 8, a grid of two tiles across, one too small for tiles
@pytest.mark.parametrize("nx,ny,count,in_place", [(512, 64, 230001, False), (64, 64, 200000, True), (32, 16, 200011, False),
                                                  (8, 64, 200003, False), (128, 32, 205000, True)])
def test_tiled_halfcell_against_short_lists(nx, ny, count, in_place):
    compare(nx, ny, count, in_place, False)


# boxes across the periodic edge (rows of 2 per cell that begin in mid-row), as wide as the grid, a last workgroup of one
# particle, less than a workgroup
@pytest.mark.parametrize("nx,ny,count,in_place", [(128, 64, 16384, False), (32, 512, 30001, True), (16, 1024, 6401, False),
                                                  (256, 32, 40, True)])
def test_boxed_halfcell_against_no_order(nx, ny, count, in_place):
    compare(nx, ny, count, in_place, True)


def compare(nx, ny, count, in_place, ordered):
    r = np.random.default_rng(nx + ny)
    dx, dy, ns, n, h = 0.5, 0.7, 6, 2, 0.25
    zs = [h * k for k in range(ns)]
    F = D((0.5 * r.standard_normal((6, ns + 2, nx * ny))).astype(np.float32))
    p = np.zeros(count, dtype=g3d_amd.PARTICLE)
    # a few boxes away on either side, and on the edge itself
    p["x"] = nx * dx * r.uniform(-0.2, 1.2, count); p["y"] = ny * dy * r.uniform(-1.1, 1.1, count)
    p["x"][:3] = (0.0, nx * dx, -nx * dx)
    if ordered:
        k = np.arange(count) + nx
        p["x"] = dx * (0.5 * k % nx + r.uniform(-0.6, 0.6, count))
        p["y"] = dy * (0.5 * k // nx + r.uniform(-0.6, 0.6, count))
    p["px"], p["py"] = 0.5 * r.standard_normal((2, count))
    p["pz"] = np.abs(r.standard_normal(count))
    p["zeta"] = zs[n + 1]; p["z"] = 20 * r.uniform(size=count) ** 6
    p["w"] = r.uniform(0.5, 1.5, count); p["q"] = -1; p["qm"] = -1; p["alive"] = 1; p["sp"] = 2
    p["id"] = np.arange(count)
    p["q"][::7] = 1
    code = r.uniform(size=count)
    p["alive"][code < 0.05] = 5; p["alive"][code > 0.9] = 6
    p["zeta"][code > 0.9] = r.uniform(zs[n] - h, zs[n + 1], (code > 0.9).sum())
    ia = np.full(ny, 1 / dy)

    def stream(lists):
        J = D(nbytes=5 * nx * ny * 8)
        sc, keep = context(nx, ny, dx, dy, F, J, zs, ia, n, ns, 0.0, 20.0)
        out = []
        for q in lists:
            src = g3d_amd.DeviceParts(q)
            dst = src if in_place else g3d_amd.DeviceParts(np.zeros_like(q))
            g3d_amd.kernel_call("g3d_stream_halfcell", C.byref(sc), C.byref(src.c), C.byref(dst.c), len(q))
            out.append(dst.records())
        return np.concatenate(out), J.get(np.float64).reshape(5, -1)

    got, Jg = stream([p])
    order = r.permutation(count) if ordered else np.arange(count)
    want, Jw = stream([p[order][k:k + SHORT] for k in range(0, count, SHORT)])
    want = want[np.argsort(order)]
    assert count < 1000 or (want["alive"] == 5).sum() > (p["alive"] == 5).sum() > 0      # the input has trapped ones
    for f in ("x", "y", "zeta", "px", "py", "pz", "z", "q", "qm", "alive"):
        assert np.array_equal(got[f], want[f]), f
    # sums of up to some thousand terms in another order
    assert np.abs(Jg - Jw).max() <= 1e-13 * np.abs(Jw).max()
