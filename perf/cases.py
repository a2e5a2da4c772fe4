"""The work that programs have this framework do, as cases that can be timed and checked.

Blocks behind the kernel-level entry points (include/g3d.h) and the autograd functions, over the caller's device
buffers, and whole runs of the engine (`g3d_amd.Sim`).  Sizes are those of the decks of bench.py and tests/decks.py
and of the grids and particle counts around them.

  halfcell  one half-cell of the streaming plasma: g3d_stream_halfcell, then g3d_stream_spectra of its current
  currents  g3d_bunch_currents: the beam deposit of a bunch and its current spectra
  sponge    g3d_sponge_real_fields: the sponge and the real fields of all slices
  march     g3d_autograd.march forward and backward: the march of all slices and its adjoint
  pushgrad  g3d_autograd.StreamPush forward and backward: the streaming push and its reverse
  run       steps of an engine deck, then the snapshot that a program takes of it (fields, beam)
  gradient  Sim.gradient on a new simulation, as an optimiser calls it
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("gem-pic-3d_amd"))

import g3d_amd  # noqa: E402
import g3d_autograd  # noqa: E402

LAMBDA0 = 2 * math.pi * 1e-6          # code units: 1 um = 1/k0
F64, C128 = torch.float64, torch.complex128


def listed():
    return [
        # the reduced laser-wakefield deck of the tests: launches and latency count
        {"name": "halfcell_32", "kind": "halfcell", "nx": 32, "ny": 32, "ppc_x": 2, "ppc_y": 2, "late": 7,
         "smooth": 0.0},
        # the transverse grid of the laser-wakefield benchmark
        {"name": "halfcell_256", "kind": "halfcell", "nx": 256, "ny": 256, "ppc_x": 2, "ppc_y": 2, "late": 1001,
         "smooth": 0.0},
        # the witness bunch of the benchmark (2^20 electrons) in a window of 128 slices
        {"name": "currents_256", "kind": "currents", "nx": 256, "ny": 256, "nz": 128, "np": 1 << 20, "sigr": 1.5,
         "sigz": 3.0, "keep0": 1, "zfilter": 1},
        # all slices of the vacuum deck
        {"name": "sponge_64", "kind": "sponge", "nx": 64, "ny": 64, "nz": 256, "sponge": 1},
        # a quarter of the window of the laser-wakefield benchmark
        {"name": "sponge_256", "kind": "sponge", "nx": 256, "ny": 256, "nz": 256, "sponge": 1},
        # gradients through the march of the vacuum deck
        {"name": "march_64", "kind": "march", "nx": 64, "ny": 64, "nz": 256, "D": 10.0},
        # the streaming push of the gradient deck (128 x 128 modes, 2 x 1 electrons per cell)
        {"name": "pushgrad_128", "kind": "pushgrad", "nx": 128, "ny": 128, "ppc_x": 2, "ppc_y": 1, "extra": 0},
        # the headline: laser wakefield at full size, FP32-mixed, four steps between snapshots of the fields
        {"name": "lwfa_mixed_256", "kind": "run", "deck": "lwfa", "n": 256, "nz": 1024, "steps": 4, "mixed": 1,
         "nmacro": 0, "ppc_x": 2, "ppc_y": 2},
        # the plain FP64 form with a witness bunch on the gradient deck's grid
        {"name": "lwfa_f64_witness_128", "kind": "run", "deck": "lwfa", "n": 128, "nz": 512, "steps": 4, "mixed": 0,
         "nmacro": 1 << 18, "ppc_x": 2, "ppc_y": 2},
        # ionization injection on the free-hand y grid (512 x 386, mobile H, N with ADK) in a short window
        {"name": "freehand_mixed_512", "kind": "run", "deck": "freehand", "n": 512, "ymax": 200.0, "Lw": 48.0,
         "steps": 2, "mixed": 1},
        # the vacuum deck: 2^18 beam electrons in the oblique plane wave
        {"name": "vacuum_64", "kind": "run", "deck": "vacuum", "n": 64, "nz": 256, "steps": 20, "mixed": 0,
         "nmacro": 1 << 18},
        # the gradient deck at the size of its tests
        {"name": "gradient_64", "kind": "gradient", "n": 64, "nz": 256, "nmacro": 16384, "steps": 2, "every": 1},
    ]


def draw(rng):
    def span(lo, hi):                 # whole numbers, even over their logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["halfcell", "halfcell", "halfcell", "currents", "currents", "sponge", "sponge", "march",
                       "pushgrad", "run", "run", "gradient"])
    if kind == "halfcell":
        return {"kind": kind, "nx": rng.choice([32, 64, 128, 256]), "ny": rng.choice([32, 64, 128, 256]),
                "ppc_x": rng.choice([1, 2, 3]), "ppc_y": rng.choice([1, 2]), "late": span(1, 3000),
                "smooth": rng.choice([0.0, 1.5])}
    if kind == "currents":
        return {"kind": kind, "nx": rng.choice([32, 64, 128, 256]), "ny": rng.choice([32, 64, 128, 256]),
                "nz": span(48, 128), "np": span(4096, 1 << 20), "sigr": rng.choice([1.5, 2.0, 4.0]),
                "sigz": rng.choice([3.0, 4.0]), "keep0": rng.choice([0, 1]), "zfilter": rng.choice([0, 1])}
    if kind == "sponge":
        return {"kind": kind, "nx": rng.choice([32, 64, 128, 256]), "ny": rng.choice([32, 64, 128, 256]),
                "nz": span(47, 256), "sponge": rng.choice([0, 1, 1])}
    if kind == "march":
        return {"kind": kind, "nx": rng.choice([32, 64, 128]), "ny": rng.choice([32, 64, 128]), "nz": span(47, 256),
                "D": rng.choice([2.5, 5.0, 10.0])}
    if kind == "pushgrad":
        return {"kind": kind, "nx": rng.choice([32, 64, 128]), "ny": rng.choice([32, 64, 128]),
                "ppc_x": rng.choice([1, 2]), "ppc_y": rng.choice([1, 2]), "extra": span(1, 999)}
    if kind == "gradient":
        return {"kind": kind, "n": rng.choice([32, 64]), "nz": rng.choice([64, 128, 256]),
                "nmacro": span(2000, 16384), "steps": rng.choice([1, 2]), "every": 1}
    deck = rng.choice(["lwfa", "lwfa", "freehand", "vacuum"])
    if deck == "lwfa":
        mixed = rng.choice([0, 1])
        return {"kind": kind, "deck": deck, "n": rng.choice([64, 128, 256]), "nz": span(128, 512),
                "steps": rng.choice([1, 2, 4]), "mixed": mixed,
                "nmacro": 0 if mixed else rng.choice([0, span(8192, 1 << 18)]), "ppc_x": rng.choice([1, 2]),
                "ppc_y": rng.choice([1, 2])}
    if deck == "freehand":
        return {"kind": kind, "deck": deck, "n": rng.choice([128, 256, 512]), "ymax": rng.choice([60.0, 120.0, 200.0]),
                "Lw": rng.uniform(8.0, 48.0), "steps": rng.choice([1, 2]), "mixed": rng.choice([0, 1])}
    return {"kind": kind, "deck": deck, "n": rng.choice([32, 64, 128]), "nz": span(64, 256),
            "steps": rng.choice([10, 20]), "mixed": 0, "nmacro": span(4096, 1 << 18)}


# ------------------------------------------------------------------------------------------------ common pieces
DX, H = 0.9375, 0.25                  # the cells and the slice distance of the laser-wakefield benchmark


def _p(t):
    return C.c_void_p(t.data_ptr())


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _k(n, d):
    """k of the FFT order, the same with the Nyquist mode zeroed, and the filter cos^2(k d / 2) without it"""
    m = np.arange(n)
    ks = 2 * np.pi * np.where(m <= n // 2, m, m - n) / (n * d)
    kz, f = ks.copy(), np.cos(0.5 * ks * d) ** 2
    kz[n // 2] = 0
    f[n // 2] = 0
    return [torch.from_numpy(a).cuda() for a in (kz, ks, f)]


class _Grid:
    """the tables of a Fourier grid with N uniform slices and a plan, as a program keeps them"""

    def __init__(self, nx, ny, nz, smooth=0.0, keep0=1):
        self.nx, self.ny, self.N, self.nk = nx, ny, nz, nx * ny
        self.kx, self.kxs, self.fx = _k(nx, DX)
        self.ky, self.kys, self.fy = _k(ny, DX)
        self.hcg = torch.full((nz + 3,), H, dtype=F64, device="cuda")
        self.half = torch.full((nz,), 0.5, dtype=F64, device="cuda")
        self.zs = torch.arange(nz, dtype=F64, device="cuda") * H
        self.iA = torch.full((ny,), 1 / DX, dtype=F64, device="cuda")
        self.plan = g3d_amd.FftPlan(nx, ny)
        self.spec = g3d_amd.SpecCtx(nx=nx, ny=ny, ns=nz, N=nz, a=0, nk=self.nk, kx=_p(self.kx), ky=_p(self.ky),
                                    kxs=_p(self.kxs), kys=_p(self.kys), filt=_p(self.fx), filty=_p(self.fy),
                                    hcg=_p(self.hcg), wlo=_p(self.half), whi=_p(self.half), a2=smooth ** 2,
                                    keep0=keep0, plan=self.plan.h.value)
        self.zax = g3d_amd.Axis(X=_p(self.zs), n=nz, uniform=1, x0=0.0, ih=1 / H)


def _filter(nx, ny, keep0, a2=0.0):
    _, kxs, fx = _k(nx, DX)
    _, kys, fy = _k(ny, DX)
    f = fx[None, :] * fy[:, None] / (1 + a2 * (kxs[None, :] ** 2 + kys[:, None] ** 2))
    if not keep0:
        f[0, 0] = 0
    return f


def _parts(cols):
    """g3d_parts over tensors"""
    return g3d_amd.Parts(**{f: cols[f].data_ptr() for f in g3d_amd.SOA_FIELDS})


def _smooth_planes(g, n, ny, nx, amp):
    """n real planes of a few low modes each"""
    y = torch.arange(ny, dtype=F64, device="cuda") * (2 * math.pi / ny)
    x = torch.arange(nx, dtype=F64, device="cuda") * (2 * math.pi / nx)
    out = torch.zeros(n, ny, nx, dtype=F64, device="cuda")
    for kx, ky in ((1, 0), (0, 1), (2, 1), (1, 3), (5, 2), (9, 4)):
        c = torch.randn(n, 2, dtype=F64, device="cuda", generator=g) * (amp / math.sqrt(6.0))
        ph = kx * x[None, :] + ky * y[:, None]
        out += c[:, 0, None, None] * torch.cos(ph) + c[:, 1, None, None] * torch.sin(ph)
    return out


def _stream_list(g, nx, ny, px, py, s0, s1, zn, zn1, late, extra):
    """The streaming electrons in the wake: the lattice of a step in the order a program loads it, displaced by up
    to a few cells, with the momenta of a wave of a0 ~ 1; some have run on almost to the end of the step, a few
    have left the stream; at the end of the list `late` electrons that wait to join at their own zeta, `extra` more
    anywhere."""
    j, i, b, a = torch.meshgrid(*[torch.arange(m, device="cuda") for m in (ny, nx, py, px)], indexing="ij")
    x = (i + (a + 0.5) / px).reshape(-1) * DX
    y = (j + (b + 0.5) / py).reshape(-1) * DX
    n = x.numel() + late + extra
    r = lambda: torch.randn(n, dtype=F64, device="cuda", generator=g)
    u = lambda: torch.rand(n, dtype=F64, device="cuda", generator=g)
    xs, ys = u() * (nx * DX), u() * (ny * DX)
    m = x.numel()
    drift_x, drift_y = _smooth_planes(g, 2, ny, nx, 0.8).reshape(2, -1)
    cell = (j * nx + i).reshape(-1)
    xs[:m] = x + drift_x[cell]
    ys[:m] = y + drift_y[cell]
    xs, ys = torch.remainder(xs, nx * DX), torch.remainder(ys, ny * DX)
    pz = 0.3 * r().abs()
    alive = torch.ones(n, dtype=torch.int32, device="cuda")
    alive[:m][u()[:m] < 1e-3] = 5
    zeta = torch.full((n,), zn1, dtype=F64, device="cuda")
    alive[m:m + late] = 6
    zeta[m:m + late] = (zn + (zn1 - zn) * (2 * u() - 0.5))[m:m + late].clamp(max=zn1)
    return {"x": xs, "y": ys, "zeta": zeta, "px": 0.4 * r(), "py": 0.3 * r(), "pz": pz,
            "w": 1e-3 * DX * DX * (s1 - s0) / (px * py) * (1 + 0.1 * u()), "z": s0 + (s1 - s0) * u() ** 8,
            "q": torch.full((n,), -1.0, dtype=F64, device="cuda"),
            "qm": torch.full((n,), -1.0, dtype=F64, device="cuda"), "rem": torch.zeros(n, dtype=F64, device="cuda"),
            "alive": alive, "sp": torch.full((n,), 2, dtype=torch.int32, device="cuda"),
            "id": torch.arange(n, dtype=torch.int64, device="cuda")}


def _tsc(xi):
    i0 = torch.floor(xi.detach() + 0.5)
    f = xi - i0
    return i0.to(torch.int64), (0.5 * (0.5 - f) ** 2, 0.75 - f * f, 0.5 * (0.5 + f) ** 2)


def _stencil(x, y, nx, ny):
    ix, wx = _tsc(x / DX)
    jy, wy = _tsc(y / DX)
    return [(torch.remainder(jy + v - 1, ny) * nx + torch.remainder(ix + u - 1, nx), wx[u] * wy[v])
            for v in range(3) for u in range(3)]


def _boris(u, E, B, qm, dt):
    qh = 0.5 * qm * dt
    a = [u[k] + qh * E[k] for k in range(3)]
    gm = torch.sqrt(1 + a[0] ** 2 + a[1] ** 2 + a[2] ** 2)
    t = [qh * B[k] / gm for k in range(3)]
    t2 = t[0] ** 2 + t[1] ** 2 + t[2] ** 2
    cross = lambda p, q: [p[1] * q[2] - p[2] * q[1], p[2] * q[0] - p[0] * q[2], p[0] * q[1] - p[1] * q[0]]
    c = cross(a, t)
    p = [a[k] + c[k] for k in range(3)]
    s = cross(p, t)
    sf = 2 / (1 + t2)
    return [a[k] + sf * s[k] + qh * E[k] for k in range(3)]


def _stream_exact(s, F0, F1, nx, ny, n, s0, s1, vz_beam):
    """the streaming push of src/sim_stream.hpp:104-171 for electrons in plain torch: the state after half-cell n and
    the current planes [5, nk]"""
    zn, zn1, Delta = n * H, (n + 1) * H, s1 - s0
    alive, zeta = s["alive"], s["zeta"]
    live = (alive == 1) | ((alive == 6) & (zeta > zn))
    full = zeta >= zn1 - 1e-9 * H
    hl = torch.where(full, torch.full_like(zeta, H), torch.clamp(zeta - zn, min=0.0))
    hl = torch.where(live, hl, torch.zeros_like(hl))
    p = [s["px"], s["py"], s["pz"]]
    pt2 = 1 + p[0] ** 2 + p[1] ** 2
    g0 = torch.sqrt(pt2 + p[2] ** 2)
    omv0 = pt2 / (g0 * (g0 + p[2]))
    dt0 = hl / omv0
    xm, ym = s["x"] + 0.5 * dt0 * p[0] / g0, s["y"] + 0.5 * dt0 * p[1] / g0
    fz = torch.where(live, (zeta - 0.5 * hl) / H - n, torch.zeros_like(zeta))
    st = _stencil(xm, ym, nx, ny)
    v0 = sum(w * F0[:, k] for k, w in st)
    v1 = sum(w * F1[:, k] for k, w in st)
    f = (1 - fz) * v0 + fz * v1
    E, B = f[:3], f[3:]
    qm = s["qm"]
    gam = lambda u: torch.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    u = _boris(p, E, B, qm, dt0)
    g1 = gam(u)
    dt = 2 * hl / (omv0 + (1 + u[0] ** 2 + u[1] ** 2) / (g1 * (g1 + u[2])))
    u = _boris(p, E, B, qm, dt)
    g1 = gam(u)
    v = [0.5 * (p[k] / g0 + u[k] / g1) for k in range(3)]
    trap = live & (s["z"] + v[2] * dt >= s1)
    dtp = torch.clamp((s1 - s["z"]) / torch.clamp(v[2], min=1e-3), min=0.0)
    dt = torch.where(trap, dtp, dt)
    ut = _boris(p, E, B, qm, dt)
    u = [torch.where(trap, ut[k], u[k]) for k in range(3)]
    g1 = gam(u)
    v = [0.5 * (p[k] / g0 + u[k] / g1) for k in range(3)]
    x, y = s["x"] + v[0] * dt, s["y"] + v[1] * dt
    keep = lambda new, old: torch.where(live, new, old)
    out = {"x": keep(x, s["x"]), "y": keep(y, s["y"]),
           "z": keep(torch.where(trap, torch.full_like(x, s1), s["z"] + v[2] * dt), s["z"]),
           "zeta": keep(torch.where(trap, zeta - (1 - v[2]) * dt, torch.full_like(x, zn)), zeta),
           "px": keep(u[0], p[0]), "py": keep(u[1], p[1]), "pz": keep(u[2], p[2]),
           "alive": torch.where(trap, torch.full_like(alive, 5), torch.where(live, torch.ones_like(alive), alive))}
    J = [torch.zeros(nx * ny, dtype=F64, device=x.device) for _ in range(4)]

    def deposit(xd, yd, c, vel, on):
        for k, w in _stencil(xd, yd, nx, ny):
            val = torch.where(on, c * w / DX, torch.zeros_like(w))
            for q in range(3):
                J[q] = J[q].index_add(0, k, val * vel[q])
            J[3] = J[3].index_add(0, k, val)

    deposit(0.5 * (s["x"] + x), 0.5 * (s["y"] + y), s["q"] * s["w"] * dt / (Delta * H * DX), v, live)
    vze = u[2] / g1
    join = trap & (vze >= vz_beam)
    deposit(x, y, s["q"] * s["w"] / (H * DX * torch.where(join, vze, torch.ones_like(vze))),
            [u[0] / g1, u[1] / g1, vze], join)
    return out, torch.stack(J + [torch.zeros_like(J[0])])


# ------------------------------------------------------------------------------------------------ half-cell
SLICES, CELL, S0, S1, VZ_BEAM = 8, 4, 20.0, 40.0, 0.9
STATE = ("x", "y", "zeta", "px", "py", "pz", "z", "alive")


def _halfcell_inputs(c, seed):
    g = _gen(seed)
    nx, ny = c["nx"], c["ny"]
    F = torch.zeros(6, SLICES + 2, ny * nx, dtype=torch.float32, device="cuda")
    for n in range(SLICES):
        F[:, n] = _smooth_planes(g, 6, ny, nx, 0.5).reshape(6, -1).float()
    cols = _stream_list(g, nx, ny, c["ppc_x"], c["ppc_y"], S0, S1, CELL * H, (CELL + 1) * H, c["late"], 0)
    return F, cols


def _halfcell_prepare(c, seed):
    F, cols = _halfcell_inputs(c, seed)
    nx, ny = c["nx"], c["ny"]
    G = _Grid(nx, ny, SLICES, smooth=c["smooth"])
    dst = {k: v.clone() for k, v in cols.items()}
    J = torch.zeros(5 * G.nk, dtype=F64, device="cuda")
    pc = g3d_amd.PushCtx(F=_p(F), a=0, ns=SLICES, N=SLICES, nx=nx, ny=ny, self=1, yf=1, nk=G.nk, dx=DX, dy=DX,
                         Lx=nx * DX, Ly=ny * DX, zax=G.zax,
                         yax=g3d_amd.Axis(X=None, n=ny + 1, uniform=1, x0=0.0, ih=1 / DX), X0=-0.5 * nx * DX,
                         Y0=-0.5 * ny * DX, zc=0.0, dz_push=S1 - S0, push_phase=0.05, zhand=-1e300,
                         zmax=(SLICES - 1) * H, ylo=-1e300, yhi=1e300, s1=S1, vz_min=0.8, hmin=H, freeze=0)
    sc = g3d_amd.StreamCtx(pc=pc, zs=_p(G.zs), J=_p(J), ia=_p(G.iA), id=_p(G.iA), Delta=S1 - S0, s1=S1, sTrap=S1,
                           vz_beam=VZ_BEAM, n=CELL)
    jsn = torch.zeros(3, G.nk, dtype=C128, device="cuda")
    scratch = torch.zeros(6 * G.nk, dtype=C128, device="cuda")
    return {"kind": "halfcell", "keep": (F, cols, G), "sc": sc, "spec": G.spec, "src": _parts(cols),
            "dst": _parts(dst), "out": dst, "n": cols["x"].numel(), "J": J, "jsn": jsn, "scratch": scratch}


def _halfcell_run(s):
    g3d_amd.kernel_call("g3d_stream_halfcell", C.byref(s["sc"]), C.byref(s["src"]), C.byref(s["dst"]), s["n"])
    g3d_amd.kernel_call("g3d_stream_spectra", C.byref(s["spec"]), _p(s["J"]), _p(s["jsn"]), _p(s["scratch"]))
    return {**{k: s["out"][k] for k in STATE}, "jsn": s["jsn"]}


def _halfcell_exact(c, seed):
    F, cols = _halfcell_inputs(c, seed)
    nx, ny = c["nx"], c["ny"]
    out, J = _stream_exact(cols, F[:, CELL].double(), F[:, CELL + 1].double(), nx, ny, CELL, S0, S1, VZ_BEAM)
    f = _filter(nx, ny, 1, c["smooth"] ** 2)
    return {**out, "jsn": (f * torch.fft.fft2(J[:3].reshape(3, ny, nx))).reshape(3, -1)}


# ------------------------------------------------------------------------------------------------ currents
def _bunch(c, seed):
    """a Gaussian bunch in the middle of the window, a little of it lost, in the random order it was drawn in"""
    g = _gen(seed)
    n = c["np"]
    r = lambda: torch.randn(n, dtype=F64, device="cuda", generator=g)
    z0 = 0.5 * (c["nz"] - 1) * H
    cols = {"x": 0.5 * c["nx"] * DX + c["sigr"] * r(), "y": 0.5 * c["ny"] * DX + c["sigr"] * r(),
            "zeta": z0 + c["sigz"] * r(), "px": 0.1 * r(), "py": 0.1 * r(), "pz": 200 * (1 + 1e-2 * r()),
            "w": torch.full((n,), 1e-3, dtype=F64, device="cuda") * (1 + 0.1 * torch.rand(n, dtype=F64, device="cuda",
                                                                                            generator=g)),
            "q": torch.full((n,), -1.0, dtype=F64, device="cuda")}
    cols["qm"] = cols["q"].clone()
    cols["z"] = torch.zeros_like(cols["x"])
    cols["rem"] = torch.zeros_like(cols["x"])
    alive = torch.ones(n, dtype=torch.int32, device="cuda")
    alive[torch.rand(n, device="cuda", generator=g) < 0.01] = 0
    cols["alive"] = alive
    cols["sp"] = torch.zeros_like(alive)
    cols["id"] = torch.arange(n, dtype=torch.int64, device="cuda")
    return cols


def _currents_prepare(c, seed):
    cols = _bunch(c, seed)
    G = _Grid(c["nx"], c["ny"], c["nz"], keep0=c["keep0"])
    jw = torch.zeros(3, c["nz"] + 3, G.nk, dtype=F64, device="cuda")
    jk = [torch.zeros(c["nz"] + 1, G.nk, dtype=C128, device="cuda") for _ in range(3)]
    scratch = torch.zeros((c["nz"] + 1) * G.nk, dtype=C128, device="cuda")
    return {"kind": "currents", "keep": cols, "G": G, "p": _parts(cols), "n": c["np"], "zf": c["zfilter"], "jw": jw,
            "jk": jk, "scratch": scratch}


def _currents_run(s):
    G = s["G"]
    g3d_amd.kernel_call("g3d_bunch_currents", C.byref(G.spec), C.byref(G.zax), _p(G.iA), _p(G.iA), DX, DX, s["zf"], 1,
                        C.byref(s["p"]), s["n"], _p(s["jw"]), _p(s["jk"][0]), _p(s["jk"][1]), _p(s["jk"][2]),
                        _p(s["scratch"]))
    return {"jw": s["jw"], "jkx": s["jk"][0], "jky": s["jk"][1], "jkz": s["jk"][2]}


def _currents_exact(c, seed):
    b = _bunch(c, seed)
    nx, ny, N = c["nx"], c["ny"], c["nz"]
    nk = nx * ny
    m = torch.floor(b["zeta"] / H).to(torch.int64)
    on = (b["alive"] == 1) & (m >= 0) & (m <= N - 2)
    b = {k: v[on] for k, v in b.items()}
    hw = m[on] + 2
    g = torch.sqrt(1 + b["px"] ** 2 + b["py"] ** 2 + b["pz"] ** 2)
    f = b["q"] * b["w"] / (H * DX * DX)
    ratio = [(b["px"] / g) / (b["pz"] / g), (b["py"] / g) / (b["pz"] / g), torch.ones_like(g)]
    jw = torch.zeros(3, (N + 3) * nk, dtype=F64, device="cuda")
    for k, w in _stencil(b["x"], b["y"], nx, ny):
        for q in range(3):
            jw[q].index_add_(0, hw * nk + k, f * w * ratio[q])
    jw = jw.reshape(3, N + 3, nk)
    lo, mid, hi = jw[:, 0:N + 1], jw[:, 1:N + 2], jw[:, 2:N + 3]
    v = 0.25 * lo + 0.5 * mid + 0.25 * hi if c["zfilter"] else mid.clone()
    v[:, 0] = 0
    v[:, N] = 0
    filt = _filter(nx, ny, c["keep0"])
    jk = [(filt * torch.fft.fft2(v[q].reshape(N + 1, ny, nx))).reshape(N + 1, nk) for q in range(3)]
    return {"jw": jw, "jkx": jk[0], "jky": jk[1], "jkz": jk[2]}


# ------------------------------------------------------------------------------------------------ sponge
BETA = 0.9999875                      # the beam of gamma 200
NAMES = ("Rx", "Ry", "Lx", "Ly", "Ez", "Bz")


def _spectra(g, nx, ny, planes, amp):
    """Hermitian spectra of real planes that fall off with k like those of a laser and its wake"""
    a = amp * torch.randn(planes, ny, nx, dtype=F64, device="cuda", generator=g)
    kx, _, _ = _k(nx, DX)
    ky, _, _ = _k(ny, DX)
    return (torch.fft.fft2(a) * torch.exp(-2 * (kx[None, :] ** 2 + ky[:, None] ** 2))).reshape(planes, -1)


def _sponge_inputs(c, seed):
    g = _gen(seed)
    nx, ny, N = c["nx"], c["ny"], c["nz"]
    arrs = {n: _spectra(g, nx, ny, N, 1.0 if n[0] == "R" else 0.1) for n in NAMES}
    arrs["jkz"] = _spectra(g, nx, ny, N + 1, 0.01)
    masks = []
    for n in (nx, ny):
        L = n * DX
        d = torch.arange(n, dtype=F64, device="cuda") * DX
        r = torch.clamp(1 - torch.minimum(d, L - d) / (0.1 * L), min=0.0)
        masks.append(1 - 0.1 * r * r)
    return arrs, masks


def _sponge_prepare(c, seed):
    arrs, masks = _sponge_inputs(c, seed)
    G = _Grid(c["nx"], c["ny"], c["nz"])
    F = torch.zeros(6, c["nz"] + 2, G.nk, dtype=torch.float32, device="cuda")
    scratch = torch.zeros(5 * c["nz"] * G.nk, dtype=C128, device="cuda")
    return {"kind": "sponge", "a": arrs, "masks": masks, "G": G, "F": F, "scratch": scratch, "on": c["sponge"]}


def _sponge_run(s):
    a = s["a"]
    g3d_amd.kernel_call("g3d_sponge_real_fields", C.byref(s["G"].spec), s["on"], _p(s["masks"][0]), _p(s["masks"][1]),
                        BETA, 1 - BETA * BETA, *[_p(a[n]) for n in NAMES], _p(a["jkz"]), _p(s["F"]),
                        _p(s["scratch"]))
    return {"Rx": a["Rx"], "Ry": a["Ry"], "F": s["F"]}


def _sponge_exact(c, seed):
    arrs, masks = _sponge_inputs(c, seed)
    nx, ny, N = c["nx"], c["ny"], c["nz"]
    sh = (-1, ny, nx)
    Rx, Ry = arrs["Rx"].reshape(sh), arrs["Ry"].reshape(sh)
    if c["sponge"]:
        kx, ky = _k(nx, DX)[0][None, :], _k(ny, DX)[0][:, None]
        k2 = kx ** 2 + ky ** 2
        ik2 = torch.where(k2 > 0, 1 / torch.where(k2 > 0, k2, torch.ones_like(k2)), torch.zeros_like(k2))
        j = arrs["jkz"].reshape(sh)
        rho = torch.zeros(N + 2, ny, nx, dtype=C128, device="cuda")
        rho[1:N + 1] = 0.5 * (j[:N] + j[1:])
        d2 = (1 - BETA * BETA) * (rho[2:] - 2 * rho[1:-1] + rho[:-2]) / (H * H)
        psi = (rho[1:-1] + d2 * ik2) * ik2
        del rho, d2
        bx, by = -(1 + BETA) * 1j * kx * psi, -(1 + BETA) * 1j * ky * psi
        m = masks[0][None, :] * masks[1][:, None]
        z = torch.fft.fft2(m * torch.fft.ifft2((Rx - bx) + 1j * (Ry - by)))
        zm = torch.roll(torch.flip(z, (1, 2)), (1, 1), (1, 2)).conj()
        Rx, Ry = 0.5 * (z + zm) + bx, -0.5j * (z - zm) + by
        del z, zm, bx, by, psi
    r = torch.fft.ifft2(Rx + 1j * Ry)
    l = torch.fft.ifft2((arrs["Lx"] + 1j * arrs["Ly"]).reshape(sh))
    z = torch.fft.ifft2((arrs["Ez"] + 1j * arrs["Bz"]).reshape(sh))
    F = torch.zeros(6, N + 2, nx * ny, dtype=F64, device="cuda")
    for k, v in enumerate((0.5 * (r.real + l.real), 0.5 * (r.imag + l.imag), z.real, 0.5 * (l.imag - r.imag),
                           0.5 * (r.real - l.real), z.imag)):
        F[k, :N] = v.reshape(N, -1)
    return {"Rx": Rx.reshape(N, -1), "Ry": Ry.reshape(N, -1), "F": F}


# ------------------------------------------------------------------------------------------------ march
def _march_inputs(c, seed):
    g = _gen(seed)
    nx, ny, N = c["nx"], c["ny"], c["nz"]
    leaves = [_spectra(g, nx, ny, N, a) for a in (1.0, 1.0, 0.1, 0.1)]
    leaves += [_spectra(g, nx, ny, N + 1, 0.01) for _ in range(5)]
    return leaves, [_spectra(g, nx, ny, N, 1.0) for _ in range(6)]


def _march_prepare(c, seed):
    leaves, bars = _march_inputs(c, seed)
    d = g3d_amd.Deck(LAMBDA0)
    d.c.nx = c["nx"]
    d.c.Lx = c["nx"] * DX
    d.y_uniform(c["ny"], c["ny"] * DX)
    d.zeta_uniform(c["nz"], (c["nz"] - 1) * H)
    d.set(dz=2 * c["D"], move_x=0, move_y=0)
    sim = g3d_amd.Sim(d)
    geom = g3d_autograd.MarchGeometry(sim, c["D"])
    sim.close()
    return {"kind": "march", "geom": geom, "leaves": [t.requires_grad_() for t in leaves], "bars": bars}


def _march_run(s):
    out = g3d_autograd.march(s["geom"], s["leaves"][:4], s["leaves"][4:])
    grads = torch.autograd.grad(out, s["leaves"], s["bars"])
    return {"fields": [t.detach() for t in out], "grads": list(grads)}


def _march_exact(c, seed):
    """the march of src/sim_kernels.hpp:173-210 (equal slices, weights 1/2) and its gradient by torch"""
    leaves, bars = _march_inputs(c, seed)
    leaves = [t.requires_grad_() for t in leaves]
    Rx0, Ry0, Ez0, Bz0, j0x, j0y, jkx, jky, jkz = leaves
    nx, ny, N, D = c["nx"], c["ny"], c["nz"], c["D"]
    a = 1j * _k(nx, DX)[0][None, :].expand(ny, nx).reshape(-1)
    b = 1j * _k(ny, DX)[0][:, None].expand(ny, nx).reshape(-1)
    k2 = -(a * a + b * b).real
    q, hh = 0.25 * H, 0.5 * H
    den = 1 + q * (D + q) * k2
    jx = 0.5 * ((j0x + jkx)[:-1] + (j0x + jkx)[1:])
    jy = 0.5 * ((j0y + jky)[:-1] + (j0y + jky)[1:])
    rsx = Rx0 + D * (a * Ez0 + b * Bz0) - D * jx
    rsy = Ry0 + D * (b * Ez0 - a * Bz0) - D * jy
    zero = torch.zeros_like(a)
    rx, ry, ez, bz, lx, ly = rsx[N - 1], rsy[N - 1], zero, zero, zero, zero
    out = [[t] for t in (rx, ry, ez, bz, lx, ly)]
    for n in range(N - 2, -1, -1):
        lsx = lx - q * (a * ez - b * bz) - hh * jkx[n + 1]
        lsy = ly - q * (a * bz + b * ez) - hh * jky[n + 1]
        cp = 0.5 * (a * (ry + ly) - b * (rx + lx))
        qp = -0.5 * a * (rx - lx) + 0.5 * b * (ly - ry)
        sx, sy = rsx[n], rsy[n]
        bzn = (bz - hh * cp - q * (a * (sy + lsy) - b * (sx + lsx))) / den
        ezn = (ez - hh * qp - q * (a * (lsx - sx) + b * (lsy - sy)) - H * jkz[n + 1]) / den
        rx, ry = sx + D * (a * ezn + b * bzn), sy + D * (b * ezn - a * bzn)
        lx, ly = lsx - q * (a * ezn - b * bzn), lsy - q * (a * bzn + b * ezn)
        ez, bz = ezn, bzn
        for o, t in zip(out, (rx, ry, ez, bz, lx, ly)):
            o.append(t)
    out = [torch.stack(o[::-1]) for o in out]
    grads = torch.autograd.grad(out, leaves, bars)
    return {"fields": [t.detach() for t in out], "grads": list(grads)}


# ------------------------------------------------------------------------------------------------ streaming reverse
PSTATE = ("x", "y", "zeta", "z", "px", "py", "pz")


def _pushgrad_inputs(c, seed):
    g = _gen(seed)
    nx, ny = c["nx"], c["ny"]
    F0, F1 = [_smooth_planes(g, 6, ny, nx, 0.5).reshape(-1) for _ in range(2)]
    cols = _stream_list(g, nx, ny, c["ppc_x"], c["ppc_y"], S0, S1, CELL * H, (CELL + 1) * H, 0, c["extra"])
    n = cols["x"].numel()
    bars = [torch.randn(n, dtype=F64, device="cuda", generator=g) for _ in PSTATE]
    bars.append(torch.randn(5 * nx * ny, dtype=F64, device="cuda", generator=g))
    return F0, F1, cols, bars


def _pushgrad_prepare(c, seed):
    F0, F1, cols, bars = _pushgrad_inputs(c, seed)
    hc = g3d_autograd.HalfCell(c["nx"], c["ny"], DX, DX, 0.0, H, CELL, S1 - S0, S1, S1, VZ_BEAM, 1 / DX)
    leaves = [t.requires_grad_() for t in [F0, F1] + [cols[k] for k in PSTATE]]
    return {"kind": "pushgrad", "hc": hc, "leaves": leaves, "fixed": [cols[k] for k in ("q", "qm", "w", "alive")],
            "bars": bars}


def _pushgrad_run(s):
    out = g3d_autograd.StreamPush.apply(s["hc"], *s["leaves"], *s["fixed"])
    grads = torch.autograd.grad(out, s["leaves"], s["bars"])
    return {"state": [t.detach() for t in out[:7]], "J": out[7].detach(), "grads": list(grads)}


def _pushgrad_exact(c, seed):
    F0, F1, cols, bars = _pushgrad_inputs(c, seed)
    leaves = [t.requires_grad_() for t in [F0, F1] + [cols[k] for k in PSTATE]]
    out, J = _stream_exact(cols, F0.reshape(6, -1), F1.reshape(6, -1), c["nx"], c["ny"], CELL, S0, S1, VZ_BEAM)
    outs = [out[k] for k in PSTATE] + [J.reshape(-1)]
    grads = torch.autograd.grad(outs, leaves, bars)
    return {"state": [t.detach() for t in outs[:7]], "J": outs[7].detach(), "grads": list(grads)}


# ------------------------------------------------------------------------------------------------ engine runs
AMU = 1822.888486
N_IP = (14.53413, 29.60125, 47.4453, 77.4735, 97.8901, 552.06732, 667.0461)


def _deck(c, seed):
    """the decks of bench.py, with the laser and the density of a scan around them drawn from the seed"""
    rng = np.random.default_rng(int(seed))
    d = g3d_amd.Deck(LAMBDA0)
    a_var, n_var = 1 + 0.05 * rng.uniform(-1, 1), 1 + 0.05 * rng.uniform(-1, 1)
    bunch_seed = int(rng.integers(1, 1 << 30))
    n = c["n"]
    d.c.nx = n
    if c["deck"] == "lwfa":
        h, Lx = 0.25 * 1024 / max(c["nz"], 256), 240.0
        Lw = (c["nz"] - 1) * h
        d.c.Lx = Lx
        d.y_uniform(n, Lx)
        d.zeta_uniform(c["nz"], Lw)
        d.set(dz=20.0, z_end=4000.0, sponge=24.0, sponge_y=24.0, move_x=0, move_y=0, plasma_on=1, n0=1e-3 * n_var,
              ppc_x=c["ppc_x"], ppc_y=c["ppc_y"], smooth_length=0.0, iterations=2, mixed=c["mixed"])
        d.add_grid_laser(a0=2.0 * a_var, waist=30.0, tau=15.0, zeta_c=0.78 * Lw, z_focus=0.0)
        if c["nmacro"]:
            d.set(charge=2.40e-12, gamma=200.0, sigx=1.5, sigy=1.5, sigz=3.0, emitx=1e-3, emity=1e-3, espread=0.0,
                  zeta_center=0.39 * Lw, nmacro=c["nmacro"], seed=bunch_seed)
        return d
    if c["deck"] == "freehand":
        d.c.Lx = 400.0 * n / 512
        d.y_table([0.0, 18.4, 30.4], [0.2, 0.2, 2.0], c["ymax"])
        d.zeta_table([0.0, 2.0, 4.0], [0.1, 0.1, 0.5], c["Lw"])
        Lz = float(d.zeta[-1])
        d.set(dz=5.0, z_end=1000.0, plasma_on=1, n0=1e-3 * n_var, ppc_x=2, ppc_y=1, move_x=0, sponge=8.0,
              sponge_y=8.0, iterations=2, mixed=c["mixed"])
        d.add_grid_laser(a0=2.5 * a_var, waist=25.0, tau=12.0, zeta_c=0.6 * Lz)
        d.add_ion(1.00794 * AMU, 1, 1, atoms=1.0, mobile=True, ionization=False)
        d.add_ion(14.0067 * AMU, 0, 7, atoms=0.01, mobile=True, ionization=True, ip_eV=N_IP)
        return d
    Lw = (c["nz"] - 1) * 0.5
    d.c.Lx = 1.25 * n
    d.y_uniform(n, 1.25 * n)
    d.zeta_uniform(c["nz"], Lw)
    d.set(dz=20.0, z_end=1000.0, sponge=8.0, sponge_y=8.0, move_x=1, move_y=1,
          charge=11.4014089e-12 * c["nmacro"] / 262144, gamma=1000.0, sigx=2.0, sigy=2.0, sigz=4.0, emitx=2e-4,
          emity=2e-4, espread=1e-3, zeta_center=0.5 * Lw, nmacro=c["nmacro"], seed=bunch_seed, laser_on=1, laser_pol=1,
          a0=a_var, theta=2e-3, tau=30.0, start_fwhm=0.0, stop_fwhm=0.0)
    return d


def _run_prepare(c, seed):
    sim = g3d_amd.Sim(_deck(c, seed))
    sim.init()
    # the beam is part of the snapshot in the FP64 form
    return {"kind": "run", "sim": sim, "steps": c["steps"], "beam": not c["mixed"] and c.get("nmacro", 0) > 0}


def _run_run(s):
    sim = s["sim"]
    for _ in range(s["steps"]):
        sim.step()
    out = {"F": sim.array("F")}
    if s["beam"]:
        p = sim.array("parts")
        out.update({k: p[k] for k in ("x", "y", "zeta", "px", "py", "pz", "alive")})
    return out


# ------------------------------------------------------------------------------------------------ gradient
def _gradient_prepare(c, seed):
    rng = np.random.default_rng(int(seed))
    n, nz = c["n"], c["nz"]
    Lw = (nz - 1) * 0.5 * 512 / nz
    d = g3d_amd.Deck(LAMBDA0)
    d.c.nx = n
    d.c.Lx = 120.0
    d.y_uniform(n, 120.0)
    d.zeta_uniform(nz, Lw)
    d.set(dz=10.0, z_end=10.0 * c["steps"], sponge=8.0, sponge_y=8.0, move_x=0, move_y=0, plasma_on=1, n0=2e-3,
          ppc_x=2, ppc_y=1, iterations=2, mixed=0, charge=5e-12, gamma=100.0, sigx=2.0, sigy=2.0, sigz=5.0, emitx=0.0,
          emity=0.0, espread=0.0, nmacro=c["nmacro"], seed=int(rng.integers(1, 1 << 30)))
    d.add_grid_laser(a0=1.0, waist=25.0, tau=1.0, zeta_c=Lw - 41.0, z_focus=0.0)
    d.set_envelope(0, list(1.5 + 0.05 * rng.standard_normal(32)), Lw - 72.0, 2.0)
    d.set_profile(list(1 + 0.05 * rng.standard_normal(16)), 90.0 * Lw / 255.5, 120.0 * Lw / 255.5)
    return {"kind": "gradient", "deck": d, "steps": c["steps"], "every": c["every"]}


def _gradient_run(s):
    sim = g3d_amd.Sim(s["deck"])
    loss, genv, gprof = sim.gradient(s["steps"], every=s["every"])
    sim.close()
    return {"loss": loss, "env": genv, "profile": gprof}


# ------------------------------------------------------------------------------------------------ interface
_PREPARE = {"halfcell": _halfcell_prepare, "currents": _currents_prepare, "sponge": _sponge_prepare,
            "march": _march_prepare, "pushgrad": _pushgrad_prepare, "run": _run_prepare,
            "gradient": _gradient_prepare}
_RUN = {"halfcell": _halfcell_run, "currents": _currents_run, "sponge": _sponge_run, "march": _march_run,
        "pushgrad": _pushgrad_run, "run": _run_run, "gradient": _gradient_run}
_EXACT = {"halfcell": _halfcell_exact, "currents": _currents_exact, "sponge": _sponge_exact, "march": _march_exact,
          "pushgrad": _pushgrad_exact}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    """None for the engine's runs: a particle march in plain numpy or torch takes far longer than 20 seconds"""
    f = _EXACT.get(case["kind"])
    return f(case, seed) if f else None


# Operations of one particle through a half-cell (gather of six components 285, two Boris rotations 160, velocities
# 60, deposit 100), of one RK4 sub-step of a beam particle, and of a complex 2D transform
PUSH_FLOP, RK4_FLOP = 605.0, 1492.0


def _fft_flop(nx, ny):
    return 5.0 * nx * ny * math.log2(nx * ny)


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("halfcell", "currents", "sponge", "march", "pushgrad"):
        nk = c["nx"] * c["ny"]
    if kind == "halfcell":
        n = nk * c["ppc_x"] * c["ppc_y"] + c["late"]
        return {"bytes": n * 148.0 + nk * (48.0 + 48.0), "flops": n * PUSH_FLOP + 1.5 * _fft_flop(c["nx"], c["ny"])}
    if kind == "currents":
        N = c["nz"]
        return {"bytes": c["np"] * 68.0 + nk * (24.0 * (N + 3) + 48.0 * (N + 1)),
                "flops": c["np"] * 120.0 + (N + 1) * (1.5 * _fft_flop(c["nx"], c["ny"]) + 20.0 * nk)}
    if kind == "sponge":
        N, on = c["nz"], c["sponge"]
        return {"bytes": nk * N * (96.0 + 24.0 + (48.0 if on else 0.0)),
                "flops": N * ((5 if on else 3) * _fft_flop(c["nx"], c["ny"]) + 60.0 * nk)}
    if kind == "march":
        N = c["nz"]
        # forward: four fields and five currents in, six fields out; backward: six adjoints in, nine out
        return {"bytes": 16.0 * nk * N * (9 + 6 + 6 + 9), "flops": 600.0 * nk * N}
    if kind == "pushgrad":
        n = nk * c["ppc_x"] * c["ppc_y"] + c["extra"]
        # forward: state, q, qm, w, alive in, state out; backward: seven adjoints in, seven out; fields and J
        return {"bytes": n * (84.0 + 56.0 + 56.0 + 56.0) + nk * 8.0 * (12 + 5 + 5 + 12),
                "flops": n * PUSH_FLOP * 4}
    if kind == "gradient":
        n, N = c["n"], c["nz"]
        # init and the steps twice (the second time with a tape) and the reverse at about twice a step
        per = 2 * (N - 1) * n * n * (2 * 64.0 + 36.0 + 384.0)
        return {"bytes": c["steps"] * 4 * per, "flops": c["steps"] * 4 * 2 * (N - 1) * n * n * (2 * PUSH_FLOP + 400.0)}
    n, steps = c["n"], c["steps"]
    if c["deck"] == "vacuum":
        N, nk = c["nz"], n * n
        per_nk = 96.0 + 80.0 + 72.0 + 120.0 + 48.0
        return {"bytes": steps * (c["nmacro"] * 172.0 + nk * N * per_nk) + nk * N * 24.0,
                "flops": steps * (c["nmacro"] * (RK4_FLOP + 120.0) + N * (6.5 * _fft_flop(n, n) + 400.0 * nk))}
    if c["deck"] == "lwfa":
        N, ny, ppc, beam = c["nz"], n, c["ppc_x"] * c["ppc_y"], c["nmacro"]
        push = 64.0 if c["mixed"] else 98.0
    else:
        # the nodes of the graded tables; electrons and two ion species at 2 x 1 per cell
        ny = 2 * int(round(92 + 15.35 + max(0.0, c["ymax"] - 30.4) / 2.0))
        N, ppc, beam, push = int(round(26 + max(0.0, c["Lw"] - 4.0) / 0.5)), 6, 0, 98.0
    nk = n * ny
    # per half-cell and pass: every streaming particle pushed, the fields gathered and the current deposited; per
    # half-cell and step: the modes' fields and currents
    per = 2 * (ppc * push + 36.0) + 384.0
    flop = 2 * (ppc * PUSH_FLOP + 5.0 * 4.5 * math.log2(nk) + 150.0)
    return {"bytes": steps * (nk * N * per + beam * 172.0) + nk * N * 24.0,
            "flops": steps * (nk * N * flop + beam * (RK4_FLOP + 120.0))}
