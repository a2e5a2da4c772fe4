// The per-mode march as two independent real systems.  a = i k_x and b = i k_y are pure imaginary and every other
// coefficient is real, so the real parts of R, L and the transverse currents couple only to the imaginary parts of
// E_z, B_z and jk_z (half 0), and the other way round (half 1).  A lane that runs one half does a third of the complex
// form's arithmetic (which multiplies by the zero real parts of a and b) with the same operands in the same order:
// a product with i k is -k x or +k x exactly, so the results are those of march_mode and march_mode_adj bit for bit
// (up to the sign of a zero).  In memory half s of R, L, j_x, j_y is the double 2 i + s of mode i, of E_z, B_z, j_z
// the double 2 i + 1 - s.
#pragma once
#include "g3d_march.hpp"

namespace g3d {

__device__ __forceinline__ double* dbl(cx* p) { return reinterpret_cast<double*>(p); }
__device__ __forceinline__ const double* dbl(const cx* p) { return reinterpret_cast<const double*>(p); }

// i k_x, i k_y of a half: acting on E_z, B_z (xe, ye; giving a part of R, L) and on R, L (xr, yr)
struct HalfK { double xe, ye, xr, yr, k2; };
__device__ __forceinline__ HalfK half_k(int half, double kx, double ky) {
    const double k2 = kx * kx + ky * ky;
    return half ? HalfK{kx, ky, -kx, -ky, k2} : HalfK{-kx, -ky, kx, ky, k2};
}
struct Half6 { double Rx, Ry, Ez, Bz, Lx, Ly; };

// den = 1 + h/4 (D + h/4) k^2 and its reciprocal, formed when h changes; div(x) = x / den: the quotient estimate
// corrected by its exact remainder, as the compiler's division does after its reciprocal, with div_fixup for infinities
// and NaN.  Scaling is left out: den is at least 1 and x a field (a quotient below 1e-290 may differ in its last bit)
struct HalfDen {
    double h = __builtin_nan(""), den = 1, r = 1;       // no step yet: NaN equals none
    __device__ __forceinline__ void set(const HalfK& k, double hn, double D) {
        if (hn == h) return;
        h = hn;
        const double qh = 0.25 * h;
        den = 1 + qh * (D + qh) * k.k2;
        r = 1 / den;
    }
    __device__ __forceinline__ double div(double x) const {
        const double q = x * r;
        const double e = fma(-q, den, x);
        return __builtin_amdgcn_div_fixup(fma(e, r, q), den, x);
    }
};

// the explicit parts R_s = R + D (F - J) of slice n (currents [0] of half-cell n-1, [1] of half-cell n)
__device__ __forceinline__ void half_explicit(const HalfK& k, double D, double wl, double wu, double Rx, double Ry,
                                              double Ez, double Bz, const double j0x[2], const double j0y[2],
                                              const double jkx[2], const double jky[2], double& Rsx, double& Rsy) {
    const double Jx = wl * (j0x[0] + jkx[0]) + wu * (j0x[1] + jkx[1]);
    const double Jy = wl * (j0y[0] + jky[0]) + wu * (j0y[1] + jky[1]);
    Rsx = Rx + D * (k.xe * Ez + k.ye * Bz) - D * Jx;
    Rsy = Ry + D * (k.ye * Ez - k.xe * Bz) - D * Jy;
}
// slice n from its explicit parts, the currents of half-cell n and slice n+1 (the implicit part of march_mode_k)
__device__ __forceinline__ Half6 half_implicit(const HalfK& k, const HalfDen& dn, double D, double h, double Rsx,
                                               double Rsy, double jx, double jy, double jz, const Half6& u) {
    const double qh = 0.25 * h, hh = 0.5 * h;
    const double Lsx = u.Lx - qh * (k.xe * u.Ez - k.ye * u.Bz) - hh * jx;
    const double Lsy = u.Ly - qh * (k.xe * u.Bz + k.ye * u.Ez) - hh * jy;
    const double Cp = 0.5 * (k.xr * (u.Ry + u.Ly) - k.yr * (u.Rx + u.Lx));
    const double Qp = -0.5 * (k.xr * (u.Rx - u.Lx)) + 0.5 * (k.yr * (u.Ly - u.Ry));
    const double SB = k.xr * Rsy + k.xr * Lsy - k.yr * Rsx - k.yr * Lsx;
    const double SE = -(k.xr * Rsx) + k.xr * Lsx + k.yr * Lsy - k.yr * Rsy;
    const double B = dn.div(u.Bz - hh * Cp - qh * SB);
    const double E = dn.div(u.Ez - hh * Qp - qh * SE - h * jz);
    return Half6{Rsx + D * (k.xe * E + k.ye * B), Rsy + D * (k.ye * E - k.xe * B), E, B,
                 Lsx - qh * (k.xe * E - k.ye * B), Lsy - qh * (k.xe * B + k.ye * E)};
}

// The transpose (march_mode_adj): given the adjoint r of slice n's outputs, the adjoints o of its level-s0 R_x, R_y,
// E_z, B_z, u of slice n+1 and the currents (d: half-cell n-1, u: n).  conj(a) = -a, conj(b) = -b.
struct HalfAdjJ { double x_d, y_d, j0x_u, j0y_u, jkx_u, jky_u, jkz_u; };     // x_d: j0_x and jk_x of half-cell n-1
__device__ __forceinline__ void half_adjoint(const HalfK& k, const HalfDen& dn, double D, double h, double wl, double wu,
                                             bool front, const Half6& r, Half6& o, Half6& u, HalfAdjJ& J) {
    double Rsx = r.Rx, Rsy = r.Ry;
    u = Half6{};
    J = HalfAdjJ{};
    if (!front) {
        const double qh = 0.25 * h, hh = 0.5 * h;
        double Lsx = r.Lx, Lsy = r.Ly;
        const double Ezb = r.Ez - D * (k.xr * r.Rx) - D * (k.yr * r.Ry) + qh * (k.xr * r.Lx) + qh * (k.yr * r.Ly);
        const double Bzb = r.Bz - D * (k.yr * r.Rx) + D * (k.xr * r.Ry) - qh * (k.yr * r.Lx) + qh * (k.xr * r.Ly);
        const double te = dn.div(Ezb), tb = dn.div(Bzb);
        u.Ez = te; u.Bz = tb;
        const double Qpb = -hh * te, SEb = -qh * te, Cpb = -hh * tb, SBb = -qh * tb;
        J.jkz_u = -h * te;
        Rsx = Rsx + k.xe * SEb + k.ye * SBb;
        Rsy = Rsy + k.ye * SEb - k.xe * SBb;
        Lsx = Lsx - k.xe * SEb + k.ye * SBb;
        Lsy = Lsy - k.ye * SEb - k.xe * SBb;
        const double qa = -0.5 * (k.xe * Qpb), qb = -0.5 * (k.ye * Qpb), ca = -0.5 * (k.xe * Cpb), cb = -0.5 * (k.ye * Cpb);
        u.Rx = -qa - cb;
        u.Lx = qa - cb;
        u.Ly = qb + ca;
        u.Ry = -qb + ca;
        u.Lx = u.Lx + Lsx;
        u.Ly = u.Ly + Lsy;
        u.Ez = u.Ez + qh * (k.xr * Lsx) + qh * (k.yr * Lsy);
        u.Bz = u.Bz - qh * (k.yr * Lsx) + qh * (k.xr * Lsy);
        J.jkx_u = -hh * Lsx;
        J.jky_u = -hh * Lsy;
    }
    o.Rx = Rsx; o.Ry = Rsy;
    o.Ez = -D * (k.xr * Rsx) - D * (k.yr * Rsy);
    o.Bz = -D * (k.yr * Rsx) + D * (k.xr * Rsy);
    o.Lx = o.Ly = 0;
    const double Jxb = -D * Rsx, Jyb = -D * Rsy;
    J.x_d = wl * Jxb; J.j0x_u = wu * Jxb; J.jkx_u = J.jkx_u + wu * Jxb;
    J.y_d = wl * Jyb; J.j0y_u = wu * Jyb; J.jky_u = J.jky_u + wu * Jyb;
}

}  // namespace g3d
