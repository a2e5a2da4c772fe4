"""The staged march and its adjoint (two real half-systems per mode) on grids and slice counts that leave remainders."""
import ctypes as C
import math

import pytest

import g3d_amd

pytestmark = pytest.mark.gpu


def march_deck(nx, ny, nz):
    d = g3d_amd.Deck(2 * math.pi * 1e-6)
    d.c.nx = nx; d.c.Lx = 0.9 * nx
    d.y_uniform(ny, 1.1 * ny)
    d.zeta_table([0.0, 2.0, 4.0], [0.2, 0.3, 0.5], nz)
    return d.set(dz=5.0, move_x=0, move_y=0)


@pytest.mark.parametrize("nx,ny,Lw", [(4, 4, 1.3), (8, 4, 2.0), (16, 16, 3.1), (64, 32, 4.7), (128, 128, 2.6)])
def test_staged_march_and_adjoint(monkeypatch, nx, ny, Lw):
    """slices of several widths: the staged march (real half-systems) against the plain one (complex), bit for bit, and
    <w, M v> = <M^T w, v> for its adjoint"""
    import torch
    import g3d_autograd
    sim = g3d_amd.Sim(march_deck(nx, ny, Lw))
    geom = g3d_autograd.MarchGeometry(sim, 2.5)
    g = torch.Generator(device="cuda").manual_seed(nx)
    ns, nk = geom.ns, geom.nk
    mk = lambda rows: torch.randn(rows, nk, dtype=torch.complex128, device="cuda", generator=g)
    old, cur = [mk(ns) for _ in range(4)], [mk(ns + 1) for _ in range(5)]
    out = {}
    for staged in ("0", "1"):
        monkeypatch.setenv("G3D_MARCH_STAGED", staged)
        leaves = [t.clone().requires_grad_() for t in old + cur]
        f = g3d_autograd.march(geom, leaves[:4], leaves[4:])
        out[staged] = [t.detach() for t in f]
    for a, b in zip(out["0"], out["1"]):
        assert torch.equal(a, b)
    w = [mk(ns) for _ in f]
    grads = torch.autograd.grad(f, leaves, w)
    dot = lambda a, b: sum(float((x.conj() * y).real.sum()) for x, y in zip(a, b))
    lhs, rhs = dot(w, out["1"]), dot(grads, old + cur)
    scale = math.sqrt(dot(w, w) * dot(out["1"], out["1"]))
    assert abs(lhs - rhs) <= 1e-13 * scale


def arrays(geom, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda rows: torch.randn(rows, geom.nk, dtype=torch.complex128, device="cuda", generator=g)
    return mk


def test_first_step_of_minus_one(monkeypatch):
    """a march against zeta (D < 0) whose steps are -1 from the first slice on: the denominators are those of that step,
    staged as plain, and the adjoint is the transpose"""
    import torch
    import g3d_autograd
    sim = g3d_amd.Sim(march_deck(8, 4, 2.0))
    geom = g3d_autograd.MarchGeometry(sim, -1.0)
    geom.tables["hcg"].fill_(-1.0)
    mk = arrays(geom, 5)
    old, cur = [mk(geom.ns) for _ in range(4)], [mk(geom.ns + 1) for _ in range(5)]
    out = {}
    for staged in ("0", "1"):
        monkeypatch.setenv("G3D_MARCH_STAGED", staged)
        leaves = [t.clone().requires_grad_() for t in old + cur]
        f = g3d_autograd.march(geom, leaves[:4], leaves[4:])
        out[staged] = [t.detach() for t in f]
    for a, b in zip(out["0"], out["1"]):
        assert torch.isfinite(torch.view_as_real(a)).all() and torch.equal(a, b)
    w = [mk(geom.ns) for _ in f]
    grads = torch.autograd.grad(f, leaves, w)
    dot = lambda a, b: sum(float((x.conj() * y).real.sum()) for x, y in zip(a, b))
    # 10 slices of some 100 roundings of 1.1e-16 on either side
    scale = math.sqrt(dot(w, w) * dot(out["1"], out["1"])) + math.sqrt(dot(grads, grads) * dot(old + cur, old + cur))
    assert geom.ns == 10 and abs(dot(w, out["1"]) - dot(grads, old + cur)) <= 1e-13 * scale


@pytest.mark.parametrize("nx,ny,cut", [(8, 4, 1), (16, 16, 4), (16, 16, 8), (8, 8, 7)])
def test_window_in_two_parts(nx, ny, cut):
    """the march of [cut, N) and then [0, cut), whose first slice takes slice cut as it stands, and the adjoint of [0, cut)
    and then [cut, N) with `up` added to the adjoint of slice cut: bit for bit the calls over [0, N)"""
    import torch
    import g3d_autograd as ga
    sim = g3d_amd.Sim(march_deck(nx, ny, 2.6))
    geom = ga.MarchGeometry(sim, 2.5)
    N, nk, lib = geom.N, geom.nk, g3d_amd.lib()
    assert N % 6 and N % 3 and 0 < cut < N - 1
    mk = arrays(geom, nx + cut)
    fields, cur, bars, jbars = [mk(N) for _ in range(6)], [mk(N + 1) for _ in range(5)], [mk(N) for _ in range(6)], [mk(N + 1) for _ in range(5)]

    def call(name, ctx, arrs, curs, parts, up=None):
        a, b = [t.clone() for t in arrs], [t.clone() for t in curs]
        c = ctx()
        for n, t in list(zip(ga._FIELDS, a)) + list(zip(ga._CURRENTS, b)):
            setattr(c, n, t.data_ptr())
        geom._common(c)
        if ctx is ga.MarchCtx:
            c.b = N
        for lo, hi in parts:
            if ctx is ga.MarchAdjCtx:
                c.up = up.data_ptr() if hi < N else None
            torch.cuda.synchronize()
            g3d_amd.check(getattr(lib, name)(C.byref(c), lo, hi))
            g3d_amd.check(lib.g3d_sync())
            if ctx is ga.MarchAdjCtx and hi < N:
                for t, u in zip(a, up):
                    t[hi] += u
        return a + b

    for got, want in zip(call("g3d_march", ga.MarchCtx, fields, cur, [(cut, N), (0, cut)]),
                         call("g3d_march", ga.MarchCtx, fields, cur, [(0, N)])):
        assert torch.equal(got, want)
    up = torch.zeros(6, nk, dtype=torch.complex128, device="cuda")
    for got, want in zip(call("g3d_march_adjoint", ga.MarchAdjCtx, bars, jbars, [(0, cut), (cut, N)], up),
                         call("g3d_march_adjoint", ga.MarchAdjCtx, bars, jbars, [(0, N)])):
        assert torch.equal(got, want)
    assert up.abs().max() > 0
