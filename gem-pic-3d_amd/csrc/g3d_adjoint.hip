// Adjoint (reverse-mode) kernels of the march, for gradients through it.  No counterpart in the reference.
// Here: the transposed per-mode update (below), the TSC deposit with its transpose (the gather) and the gather's
// position derivatives, and the reverse of the Boris rotation.
//
// The per-mode march of slice n (march_mode) is complex-linear in its inputs: the level-s0 values of slice n
// (R_x, R_y, E_z, B_z), the level-s1 values of slice n+1 (six), and the currents of half-cells n-1 and n.  Its
// coefficients are real (D, h/4, h/2, h, 1/den, the ζ weights) or the pure imaginary a = i k_x, b = i k_y.  For the
// real inner product <u, v> = Re Σ conj(u) v, the adjoint of v = A u is u' = A^H v', so every statement of the
// forward update is transposed in reverse order with conj(a) = -a, conj(b) = -b.  The march over slices runs front
// to rear (n = hi-1 ... lo, slice n reading slice n+1); its adjoint runs rear to front, carrying the adjoint of the
// slice n+1 values from the update of slice n to that of slice n+1.
#include "g3d_boris_rev.hpp"
#include "g3d_kernels.hpp"
#include "g3d_march_adj.hpp"
#include "g3d_march_half.hpp"
#include "g3d_runtime.hpp"

namespace g3d {
namespace {

// Slices lo ... hi-1 of every mode, rear to front: the transpose of the march.  Like k_march_staged, two lanes per
// mode (one real half-system each) and 32 modes per workgroup: wave 0 runs the chain from LDS, waves 1-3 load the next
// block of kAdjB slices (one each) into the other of two buffers and clear L_x, L_y, which are not inputs.  As one
// lane per mode with complex arithmetic and its loads on the chain it took 742 us for 64 x 64 x 256, now 143 us.  Larger grids
// are bound by the 22 planes that a slice reads and writes: 256 x 256 x 64 298 us, 512 x 512 x 32 646 us (5.0 and 4.6 TB/s).
constexpr int kAdjB = 3, kAdjComp = 11;
__global__ void __launch_bounds__(256) k_march_adj(AdjView c, int lo, int hi) {
    __shared__ double stg[2 * kAdjB * kAdjComp * 64], wts[2 * kAdjB * 3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane & 1;
    const long i = long(blockIdx.x) * 32 + (lane >> 1);
    const bool on = i < c.nk;
    const long ic = on ? i : c.nk - 1, p = 2 * ic + half, e = 2 * ic + 1 - half;
    const int nblk = (hi - lo + kAdjB - 1) / kAdjB;
    if (wave > 0) {
        double r[kAdjComp], w[3];
        const int s0 = wave - 1;
        auto load = [&](int b) {
            const int n = lo + b * kAdjB + s0;
            if (n >= hi) return;
            const long o = 2 * long(n - c.a) * c.nk;
            r[0] = dbl(c.Rx)[o + p]; r[1] = dbl(c.Ry)[o + p]; r[2] = dbl(c.Ez)[o + e]; r[3] = dbl(c.Bz)[o + e];
            r[4] = dbl(c.Lx)[o + p]; r[5] = dbl(c.Ly)[o + p];
            r[6] = dbl(c.j0x)[o + p]; r[7] = dbl(c.j0y)[o + p]; r[8] = dbl(c.jkx)[o + p]; r[9] = dbl(c.jky)[o + p];
            r[10] = dbl(c.jkz)[o + e];
            w[0] = c.wlo[n]; w[1] = c.whi[n]; w[2] = n < c.N - 1 ? c.hcg[n + 2] : 0.0;
        };
        auto write = [&](int b) {
            const int n = lo + b * kAdjB + s0, s = (b & 1) * kAdjB + s0;
            if (n >= hi) return;
#pragma unroll
            for (int q = 0; q < kAdjComp; ++q) stg[(s * kAdjComp + q) * 64 + lane] = r[q];
            if (lane < 3) wts[3 * s + lane] = w[lane];
            if (on) {
                const long o = 2 * long(n - c.a) * c.nk;
                dbl(c.Lx)[o + p] = 0; dbl(c.Ly)[o + p] = 0;
            }
        };
        load(0);
        write(0);
        if (nblk > 1) load(1);
        for (int b = 0; b < nblk; ++b) {
            __syncthreads();
            if (b + 1 < nblk) write(b + 1);
            if (b + 2 < nblk) load(b + 2);
        }
        return;
    }
    const int ixx = int(ic % c.nx), j = int(ic / c.nx);
    const HalfK k = half_k(half, c.kx[ixx], c.ky[j]);
    HalfDen dn{};
    Half6 carry{};                                  // adjoint of slice n's outputs from slice n-1's use of them
    double d0x = 0, d0y = 0, dkx = 0, dky = 0, dkz = 0;      // half-cell n-1 (plane n - a) so far
    for (int b = 0; b < nblk; ++b) {
        __syncthreads();
        for (int s = 0; s < kAdjB; ++s) {
            const int n = lo + b * kAdjB + s;
            if (n >= hi) break;
            const int sb = (b & 1) * kAdjB + s;
            const double* q = stg + sb * kAdjComp * 64 + lane;
            const double wl = wts[3 * sb], wu = wts[3 * sb + 1], h = wts[3 * sb + 2];
            const Half6 r{q[0] + carry.Rx, q[64] + carry.Ry, q[128] + carry.Ez, q[192] + carry.Bz, q[256] + carry.Lx,
                          q[320] + carry.Ly};
            const double c0x = q[384], c0y = q[448], ckx = q[512], cky = q[576], ckz = q[640];
            const bool front = n == c.N - 1;
            if (!front) dn.set(k, h, c.D);
            Half6 old;
            HalfAdjJ J;
            half_adjoint(k, dn, c.D, h, wl, wu, front, r, old, carry, J);
            if (on) {
                const long o = 2 * long(n - c.a) * c.nk;
                dbl(c.Rx)[o + p] = old.Rx; dbl(c.Ry)[o + p] = old.Ry; dbl(c.Ez)[o + e] = old.Ez; dbl(c.Bz)[o + e] = old.Bz;
                // plane n - a is half-cell n-1: the "u" currents of slice n-1 and the "d" currents of slice n
                dbl(c.j0x)[o + p] = c0x + d0x + J.x_d; dbl(c.j0y)[o + p] = c0y + d0y + J.y_d;
                dbl(c.jkx)[o + p] = ckx + dkx + J.x_d; dbl(c.jky)[o + p] = cky + dky + J.y_d;
                dbl(c.jkz)[o + e] = ckz + dkz;
            }
            d0x = J.j0x_u; d0y = J.j0y_u; dkx = J.jkx_u; dky = J.jky_u; dkz = J.jkz_u;
        }
    }
    if (!on) return;
    const long o = 2 * long(hi - c.a) * c.nk;        // plane hi - a: half-cell hi-1
    dbl(c.j0x)[o + p] += d0x; dbl(c.j0y)[o + p] += d0y; dbl(c.jkx)[o + p] += dkx; dbl(c.jky)[o + p] += dky;
    dbl(c.jkz)[o + e] += dkz;
    if (c.up && hi < c.N) {
        const long pl = 2 * c.nk;
        double* u = dbl(c.up);
        u[p] = carry.Rx; u[pl + p] = carry.Ry; u[2 * pl + e] = carry.Ez; u[3 * pl + e] = carry.Bz;
        u[4 * pl + p] = carry.Lx; u[5 * pl + p] = carry.Ly;
    }
}

// ---------------------------------------------------------------- TSC deposit and its transpose
__global__ void __launch_bounds__(256) k_tsc_deposit(g3d_tsc_ctx c, const double* q, double* plane) {
    const long p = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= c.np) return;
    int ix[3], jn[3]; double wx[3], wn[3];
    tsc_periodic(c.x[p], c.dx, c.nx, ix, wx);
    tsc_periodic(c.y[p], c.dy, c.ny, jn, wn);
    for (int v = 0; v < 3; ++v)
        for (int u = 0; u < 3; ++u) atomicAdd(&plane[long(jn[v]) * c.nx + ix[u]], wx[u] * wn[v] * q[p]);
}
// d/dx of the TSC weights of x (index coordinate xi = x/d, f = xi - round(xi)): the derivative of
// 1/2 (1/2 - f)^2, 3/4 - f^2, 1/2 (1/2 + f)^2, times 1/d
__device__ __forceinline__ void tsc_dweights(double x, double d, double dw[3]) {
    const double xi = x / d;
    const double f = xi - floor(xi + 0.5);
    dw[0] = -(0.5 - f) / d;
    dw[1] = -2 * f / d;
    dw[2] = (0.5 + f) / d;
}
__global__ void __launch_bounds__(256) k_tsc_gather(g3d_tsc_ctx c, const double* plane, double* out, double* gx,
                                                    double* gy) {
    const long p = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= c.np) return;
    int ix[3], jn[3]; double wx[3], wn[3], dx[3], dy[3];
    tsc_periodic(c.x[p], c.dx, c.nx, ix, wx);
    tsc_periodic(c.y[p], c.dy, c.ny, jn, wn);
    double s = 0, sx = 0, sy = 0;
    const bool grad = gx && gy;
    if (grad) { tsc_dweights(c.x[p], c.dx, dx); tsc_dweights(c.y[p], c.dy, dy); }
    for (int v = 0; v < 3; ++v)
        for (int u = 0; u < 3; ++u) {
            const double P = plane[long(jn[v]) * c.nx + ix[u]];
            s += wx[u] * wn[v] * P;
            if (grad) { sx += dx[u] * wn[v] * P; sy += wx[u] * dy[v] * P; }
        }
    out[p] = s;
    if (grad) { gx[p] = sx; gy[p] = sy; }
}

// ---------------------------------------------------------------- Boris rotation and its reverse
__global__ void __launch_bounds__(256) k_boris(g3d_boris_args a) {
    const long p = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= a.np) return;
    const double E[3] = {a.Ex[p], a.Ey[p], a.Ez[p]}, B[3] = {a.Bx[p], a.By[p], a.Bz[p]};
    double ux = a.ux[p], uy = a.uy[p], uz = a.uz[p];
    boris(ux, uy, uz, E, B, a.qm[p], a.dt[p]);
    a.ux[p] = ux; a.uy[p] = uy; a.uz[p] = uz;
}
// reverse mode of boris() (g3d_common.hpp): boris_rev (g3d_boris_rev.hpp)
__global__ void __launch_bounds__(256) k_boris_vjp(g3d_boris_args a, g3d_boris_adj g) {
    const long p = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= a.np) return;
    const double E[3] = {a.Ex[p], a.Ey[p], a.Ez[p]}, B[3] = {a.Bx[p], a.By[p], a.Bz[p]};
    const double u[3] = {a.ux[p], a.uy[p], a.uz[p]};
    const double ub[3] = {g.ubx[p], g.uby[p], g.ubz[p]};
    double ab[3], Eb[3] = {0, 0, 0}, Bb[3] = {0, 0, 0}, qmb = 0, dtb = 0;
    boris_rev(u, E, B, a.qm[p], a.dt[p], ub, ab, Eb, Bb, qmb, dtb);
    g.gux[p] = ab[0]; g.guy[p] = ab[1]; g.guz[p] = ab[2];
    g.gEx[p] = Eb[0]; g.gEy[p] = Eb[1]; g.gEz[p] = Eb[2];
    g.gBx[p] = Bb[0]; g.gBy[p] = Bb[1]; g.gBz[p] = Bb[2];
    g.gqm[p] = qmb;
    g.gdt[p] = dtb;
}

}  // namespace
}  // namespace g3d

extern "C" {
int g3d_tsc_deposit(const g3d_tsc_ctx* c, const double* q, double* plane) {
    return g3d::guard([&] {
        if (!c || !c->x || !c->y || !q || !plane || c->nx < 1 || c->ny < 1 || c->np < 0)
            throw std::invalid_argument("tsc deposit: bad context");
        if (c->np == 0) return;
        hipLaunchKernelGGL(g3d::k_tsc_deposit, dim3(g3d::blocks_for(c->np, 256)), dim3(256), 0, g3d::stream(), *c, q,
                           plane);
        g3d::launch_check("tsc deposit");
    });
}
int g3d_tsc_gather(const g3d_tsc_ctx* c, const double* plane, double* out, double* gx, double* gy) {
    return g3d::guard([&] {
        if (!c || !c->x || !c->y || !plane || !out || c->nx < 1 || c->ny < 1 || c->np < 0 || (!gx) != (!gy))
            throw std::invalid_argument("tsc gather: bad context");
        if (c->np == 0) return;
        hipLaunchKernelGGL(g3d::k_tsc_gather, dim3(g3d::blocks_for(c->np, 256)), dim3(256), 0, g3d::stream(), *c, plane,
                           out, gx, gy);
        g3d::launch_check("tsc gather");
    });
}
int g3d_boris(const g3d_boris_args* a) {
    return g3d::guard([&] {
        if (!a || a->np < 0) throw std::invalid_argument("boris: bad arguments");
        if (a->np == 0) return;
        hipLaunchKernelGGL(g3d::k_boris, dim3(g3d::blocks_for(a->np, 256)), dim3(256), 0, g3d::stream(), *a);
        g3d::launch_check("boris");
    });
}
int g3d_boris_vjp(const g3d_boris_args* a, const g3d_boris_adj* g) {
    return g3d::guard([&] {
        if (!a || !g || a->np < 0) throw std::invalid_argument("boris vjp: bad arguments");
        if (a->np == 0) return;
        hipLaunchKernelGGL(g3d::k_boris_vjp, dim3(g3d::blocks_for(a->np, 256)), dim3(256), 0, g3d::stream(), *a, *g);
        g3d::launch_check("boris vjp");
    });
}
int g3d_march_adjoint(const g3d_march_adj_ctx* m, int lo, int hi) {
    return g3d::guard([&] {
        if (!m || !m->Rx || !m->Ry || !m->Ez || !m->Bz || !m->Lx || !m->Ly || !m->j0x || !m->j0y || !m->jkx ||
            !m->jky || !m->jkz || !m->kx || !m->ky || !m->hcg || !m->wlo || !m->whi)
            throw std::invalid_argument("march adjoint: null pointer in the context");
        if (m->nx < 1 || m->ny < 1 || m->nk != long(m->nx) * m->ny)
            throw std::invalid_argument("march adjoint: nk must be nx * ny");
        if (lo < m->a || hi > m->N || lo >= hi)
            throw std::invalid_argument("march adjoint: need a <= lo < hi <= N");
        g3d::AdjView v;
        v.Rx = m->Rx; v.Ry = m->Ry; v.Ez = m->Ez; v.Bz = m->Bz; v.Lx = m->Lx; v.Ly = m->Ly; v.up = m->up;
        v.j0x = m->j0x; v.j0y = m->j0y; v.jkx = m->jkx; v.jky = m->jky; v.jkz = m->jkz;
        v.kx = m->kx; v.ky = m->ky; v.hcg = m->hcg; v.wlo = m->wlo; v.whi = m->whi;
        v.D = m->D; v.a = m->a; v.N = m->N; v.nx = m->nx; v.nk = m->nk;
        hipLaunchKernelGGL(g3d::k_march_adj, dim3(g3d::blocks_for(v.nk, 32)), dim3(256), 0, g3d::stream(), v, lo,
                           hi);
        g3d::launch_check("march adjoint");
    });
}
}
