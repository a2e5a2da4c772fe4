// Particle kernels: the RK4 push in z of the beam list with its gathers and the analytic laser, the beam deposit,
// the streaming half-cell pass (two Boris rotations, the deposit, trapping, ADK ionization), and the list tools.
// One lane per particle over structure-of-arrays streams.
#include <algorithm>
#include <type_traits>

#include <rocprim/device/device_radix_sort.hpp>

#include "g3d_kernels.hpp"
#include "g3d_nodebox.hpp"
#include "g3d_runtime.hpp"

namespace g3d {
namespace {
constexpr int kT = 256;

// ---------------------------------------------------------------- streaming particles (src/sim_stream.hpp)
// LDS windows of a tile, WX x WY nodes from node (x0, y0) (periodic); WX = 0 for particles without one (one copy of
// the push in the code for both):
//   lds   the 5 current planes of the deposit
//   fld   the fields of slices fl and fl+1 for the gather, node-major (3 float4 per node, win_node),
//         loaded once per workgroup instead of 108 scattered loads per particle
//   yn    free-hand y: the nodes y_lo ... y_lo + nyn of the axis, where the locates look first (a bisection of the
//         table in memory is a chain of dependent loads)
// The pointers carry the LDS address space: through generic ones the free-hand kernel with ions, which keeps part of
// its context in memory, read and added by flat instructions (439 us against 350 at 512 x 386 with H and N).
#define G3D_LDS __attribute__((address_space(3)))
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef G3D_LDS double* ldsd;
struct Win {
    ldsd lds;
    const G3D_LDS f4v* fld;
    const G3D_LDS double* yn;
    int x0, y0, WX, WY, fl, y_lo, nyn;
};
__device__ __forceinline__ void lds_add(ldsd p, double v) { atomicAdd((double*)p, v); }
// A node's 12 floats: E_x E_z B_y of slices fl, fl+1 (on the nodes of the free-hand y grid), then E_y B_x B_z of both
// (on its half-nodes), so that either group is a 16-byte and an 8-byte LDS read
__device__ __forceinline__ void win_node(G3D_LDS f4v* q, const float* src, long cs, long nk, bool in) {
    float f[12];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int comp = g == 0 ? 2 * k : (k == 0 ? 1 : 2 * k + 1);      // 0 2 4, then 1 3 5
            f[6 * g + k] = in ? src[comp * cs] : 0.0f;
            f[6 * g + 3 + k] = in ? src[comp * cs + nk] : 0.0f;
        }
#pragma unroll
    for (int k = 0; k < 3; ++k) q[k] = f4v{f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]};
}

// tsc_freehand with the cell looked up among the window's nodes first (the cell X[i] <= y < X[i+1] is unique, so the
// result is the same)
__device__ __forceinline__ void tsc_freehand_w(const Axis& ax, const Win& w, double y, int jn[3], double wn[3],
                                               int jh[3], double wh[3]) {
    int i; double f;
    if (w.nyn > 0 && w.yn[0] <= y && y < w.yn[w.nyn]) {
        int lo = 0, hi = w.nyn;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (w.yn[mid] <= y) lo = mid; else hi = mid;
        }
        i = w.y_lo + lo; f = (y - w.yn[lo]) / (w.yn[lo + 1] - w.yn[lo]);
    } else ax.locate(y, i, f);
    const double xi = i + f;
    tsc_w(xi, jn, wn);
    tsc_w(xi - 0.5, jh, wh);
}

// The TSC stencil of a point in the window: the first node (and half-node) and the weights; false when a row or
// column that the sums need lies outside it.  Free-hand y: window rows are node indices, rows beyond the walls are
// skipped (bits of skn, skh)
struct WinStencil {
    int kn, kh;
    unsigned skn, skh;
    double wx[3], wn[3], wh[3];
};
template <int YF>
__device__ __forceinline__ bool win_stencil(const FieldView& c, const Win& w, double x, double y, WinStencil& s) {
    int ix[3], jn[3], jh[3];
    tsc_periodic(x, c.dx, c.nx, ix, s.wx);
    const int u0 = wrap_index(ix[0] - w.x0, c.nx);
    if (u0 + 2 >= w.WX) return false;
    s.skn = s.skh = 0;
    if constexpr (YF == 1) {
        tsc_periodic(y, c.dy, c.ny, jn, s.wn);
        const int v0 = wrap_index(jn[0] - w.y0, c.ny);
        if (v0 + 2 >= w.WY) return false;
        s.kn = s.kh = v0 * w.WX + u0;
    } else {
        tsc_freehand_w(c.yax, w, y, jn, s.wn, jh, s.wh);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (jn[j] < 0 || jn[j] >= c.ny) s.skn |= 1u << j;
            else if (jn[j] < w.y0 || jn[j] >= w.y0 + w.WY) return false;
            if (jh[j] < 0 || jh[j] >= c.ny) s.skh |= 1u << j;
            else if (jh[j] < w.y0 || jh[j] >= w.y0 + w.WY) return false;
        }
        s.kn = (jn[0] - w.y0) * w.WX + u0;
        s.kh = (jh[0] - w.y0) * w.WX + u0;
    }
    return true;
}
// The sums of a stencil, g q(fl) + f q(fl+1) per node with the weights and in the order of gather(), so that the
// values are those of a gather from F.  TWO: also E at two further points in zeta (g1, f1 and g0, f0) from the same
// reads
template <int YF, bool TWO>
__device__ __forceinline__ void win_sums(const Win& w, const WinStencil& s, double g, double f, double E[3], double B[3],
                                         double g1, double f1, double g0, double f0, double E1[3], double E0[3]) {
    double v[6] = {0, 0, 0, 0, 0, 0}, a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        if (YF == 1 || !(s.skn >> j & 1u)) {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const G3D_LDS f4v* q = w.fld + 3 * (s.kn + j * w.WX + i);
                const double wt = s.wx[i] * s.wn[j];
                const f4v p = q[0];
                const f2v r = *(const G3D_LDS f2v*)(q + 1);
                const double x0 = p.x, z0 = p.y, x1 = p.w, z1 = r.x;
                v[0] += wt * (g * x0 + f * x1);
                v[2] += wt * (g * z0 + f * z1);
                v[4] += wt * (g * double(p.z) + f * double(r.y));
                if (TWO) {
                    a[0] += wt * (g1 * x0 + f1 * x1); a[2] += wt * (g1 * z0 + f1 * z1);
                    b[0] += wt * (g0 * x0 + f0 * x1); b[2] += wt * (g0 * z0 + f0 * z1);
                }
            }
        }
        if (YF == 1 || !(s.skh >> j & 1u)) {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const G3D_LDS f4v* q = w.fld + 3 * (s.kh + j * w.WX + i);
                const double wt = s.wx[i] * (YF == 1 ? s.wn[j] : s.wh[j]);
                const f2v r = *((const G3D_LDS f2v*)(q + 1) + 1);
                const f4v p = q[2];
                const double y0 = r.x, y1 = p.y;
                v[1] += wt * (g * y0 + f * y1);
                v[3] += wt * (g * double(r.y) + f * double(p.z));
                v[5] += wt * (g * double(p.x) + f * double(p.w));
                if (TWO) { a[1] += wt * (g1 * y0 + f1 * y1); b[1] += wt * (g0 * y0 + f0 * y1); }
            }
        }
    }
    E[0] = v[0]; E[1] = v[1]; E[2] = v[2]; B[0] = v[3]; B[1] = v[4]; B[2] = v[5];
    if (TWO)
        for (int k = 0; k < 3; ++k) { E1[k] = a[k]; E0[k] = b[k]; }
}
// the factors of slices fl and fl+1 at zeta; false when the pair is not the window's.  A point on slice fl+1 itself
// (the pair fl+1, fl+2 with f = 0) is 0 q(fl) + 1 q(fl+1): the same sum for finite fields
__device__ __forceinline__ bool win_pair(const FieldView& c, const Win& w, double zeta, double& g, double& f) {
    int n; double fz;
    c.zax.locate(zeta, n, fz);
    if (n == c.a - 1 && fz > 1 - 1e-9) { n = c.a; fz = 0; }
    g = 1 - fz; f = fz;
    if (n - c.a == w.fl) return true;
    if (n - c.a == w.fl + 1 && fz == 0) { g = 0; f = 1; return true; }
    return false;
}

// E, B from the tile's field window: false when the stencil or the slice pair is not in the window (then the caller
// gathers from F)
template <int YF>
__device__ __forceinline__ bool gather_window(const FieldView& c, const Win& w, double x, double y, double zeta,
                                              double E[3], double B[3]) {
    if (!c.self) return false;
    double g, f;
    WinStencil s;
    if (!win_pair(c, w, zeta, g, f) || !win_stencil<YF>(c, w, x, y, s)) return false;
    win_sums<YF, false>(w, s, g, f, E, B, 0, 0, 0, 0, nullptr, nullptr);
    return true;
}

// ---------------------------------------------------------------- RK4 in z (src/sim_kernels.hpp:73-149)
struct St { double x, y, zeta, px, py, pz; };

// E, B at a beam particle: from the field window of its workgroup when the stencil and the slice pair lie in it (the
// same values: the window's sums are gather's), else from F
__device__ __forceinline__ bool rhs(const PushArgs& c, const Win& win, const St& Y, double z, double qm, St& d) {
    const double g = sqrt(1 + Y.px * Y.px + Y.py * Y.py + Y.pz * Y.pz);
    if (Y.pz < 0.3 * g) return false;
    const double gm = (1 + Y.px * Y.px + Y.py * Y.py) / (g + Y.pz);
    double E[3], B[3], Ee[3], Be[3];
    const double xw = wrap_mod(Y.x, c.fv.Lx), yw = c.fv.yf ? wrap_mod(Y.y, c.fv.Ly) : Y.y;
    if (!(win.WX && gather_window<1>(c.fv, win, xw, yw, Y.zeta, E, B))) gather(c.fv, xw, yw, Y.zeta, E, B);
    c.laser.field(Y.x + c.X0, z, z - (Y.zeta - c.zc), Ee, Be);
    for (int k = 0; k < 3; ++k) { E[k] += Ee[k]; B[k] += Be[k]; }
    const double ip = 1 / Y.pz;
    d.x = Y.px * ip; d.y = Y.py * ip; d.zeta = -gm * ip;
    d.px = qm * (g * E[0] + Y.py * B[2] - Y.pz * B[1]) * ip;
    d.py = qm * (g * E[1] + Y.pz * B[0] - Y.px * B[2]) * ip;
    d.pz = qm * (g * E[2] + Y.px * B[1] - Y.py * B[0]) * ip;
    return true;
}
__device__ __forceinline__ St axpy(const St& a, double h, const St& b) {
    return St{a.x + h * b.x, a.y + h * b.y, a.zeta + h * b.zeta, a.px + h * b.px, a.py + h * b.py, a.pz + h * b.pz};
}

// beam particle ip from s0 (or from its hand-over point) to s1 (src/sim_kernels.hpp:98-149)
__device__ __forceinline__ void push_beam_one(const PushArgs& c, const Win& win, Parts P, long ip, double z0) {
    const int alive = P.alive[ip];
    if (alive != 1 && alive != 3) return;
    double z = alive == 3 ? c.s1 - P.rem[ip] : z0;
    if (c.freeze && is_bunch(P.sp[ip])) { P.z[ip] = c.s1; return; }
    St Y{P.x[ip], P.y[ip], P.zeta[ip], P.px[ip], P.py[ip], P.pz[ip]};
    const double qm = P.qm[ip];
    auto store = [&](const St& s) {
        P.x[ip] = s.x; P.y[ip] = s.y; P.zeta[ip] = s.zeta; P.px[ip] = s.px; P.py[ip] = s.py; P.pz[ip] = s.pz;
    };
    while (z < c.s1 - 1e-12 * fabs(c.s1)) {
        if (Y.zeta < c.zhand) { store(Y); P.alive[ip] = 2; P.rem[ip] = c.s1 - z; return; }
        if (c.vz_min > 0 && Y.pz < c.vz_min * sqrt(1 + Y.px * Y.px + Y.py * Y.py + Y.pz * Y.pz)) {
            store(Y); P.z[ip] = z; P.alive[ip] = 4;
            return;
        }
        double ds = c.dz_push < c.s1 - z ? c.dz_push : c.s1 - z;
        {
            const double g = sqrt(1 + Y.px * Y.px + Y.py * Y.py + Y.pz * Y.pz);
            const double lz = 0.5 * c.hmin * Y.pz * (g + Y.pz) / (1 + Y.px * Y.px + Y.py * Y.py);
            if (lz < ds) ds = (c.s1 - z) / ceil((c.s1 - z) / lz);
        }
        if (c.laser.on) {
            const double g = sqrt(1 + Y.px * Y.px + Y.py * Y.py + Y.pz * Y.pz);
            const double hl = g - Y.px * c.laser.kx - Y.pz * c.laser.kz;
            const double lim = c.push_phase * Y.pz / (c.laser.kL * (hl > 1e-12 ? hl : 1e-12));
            if (lim < ds) ds = (c.s1 - z) / ceil((c.s1 - z) / lim);
        }
        // the four stages as a loop (one copy of the gather in the code; unrolled they took 255 VGPRs and 100 KB of
        // instructions: 106 us against 115 for 2^18 electrons), the sums k1 + 2 k2 + 2 k3 + k4 from the left
        St k{}, A{};
        const double hd = 0.5 * ds;
#pragma unroll 1
        for (int st = 0; st < 4; ++st) {
            const double hs = st == 0 ? 0.0 : (st == 3 ? ds : hd);
            const St Ys = st == 0 ? Y : axpy(Y, hs, k);
            if (!rhs(c, win, Ys, z + hs, qm, k)) { P.alive[ip] = 0; return; }
            if (st == 0) A = k;
            else {
                const double m = st == 3 ? 1.0 : 2.0;
                A = St{A.x + m * k.x, A.y + m * k.y, A.zeta + m * k.zeta, A.px + m * k.px, A.py + m * k.py, A.pz + m * k.pz};
            }
        }
        const double w = ds / 6;
        Y.x += w * A.x; Y.y += w * A.y; Y.zeta += w * A.zeta; Y.px += w * A.px; Y.py += w * A.py; Y.pz += w * A.pz;
        z += ds;
    }
    store(Y);
    P.z[ip] = c.s1;
    int al = (Y.zeta < 0 || Y.zeta >= c.zmax || Y.y < c.ylo || Y.y > c.yhi) ? 0 : 1;
    if (al == 1 && Y.zeta < c.zhand) { al = 2; P.rem[ip] = 0; }
    P.alive[ip] = al;
}

__global__ void __launch_bounds__(kT) k_bunch_push(PushArgs c, Parts P, long np, double z0) {
    const long ip = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (ip >= np) return;
    push_beam_one(c, Win{}, P, ip, z0);
}

// ---- the beam push with field windows (Fourier y): the particles binned by (slice pair, transverse tile of kBT x kBT
// cells) through an index list (the list itself keeps its order), a workgroup per chunk of at most kBChunk
// particles of a bin with the bin's window of both slices in LDS (a chain of four dependent gathers per RK4 sub-step
// then waits on LDS instead of memory)
constexpr int kBT = 8, kBM = 1, kBW = kBT + 3 + 2 * kBM, kBChunk = 1024;
constexpr unsigned long long kBNone = ~0ull;
// Long lists by radix passes: the default merges up to 2^20 records (16 launches for 2^18).  The push of 8000 electrons in
// 256 slices of 64 x 64, by radix passes and merged, 100 and 69 us, 32000 121 and 97, 65000 153 and 131, 131000 165 and 157,
// 2^18 192 and 227
using BpushSort = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config, rocprim::default_config, 0>;
constexpr long kBpushMerge = 1L << 17;               // records up to which the default is used

// the bin of every particle that moves (alive 1 or 3, not frozen); the bin nbin (no window) for one outside the
// slices of F; ~0 for the others (a frozen bunch particle only takes the new z here, as the plain push does)
__global__ void __launch_bounds__(kT) k_bpush_keys(PushArgs c, Parts P, long np, int ntx, int nty, long nbin,
                                                   unsigned long long* key, unsigned* idx) {
    const long ip = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (ip >= np) return;
    idx[ip] = unsigned(ip);
    key[ip] = kBNone;
    const int alive = P.alive[ip];
    if (alive != 1 && alive != 3) return;
    if (c.freeze && is_bunch(P.sp[ip])) { P.z[ip] = c.s1; return; }
    const FieldView& F = c.fv;
    int n; double fz;
    F.zax.locate(P.zeta[ip], n, fz);
    if (n == F.a - 1 && fz > 1 - 1e-9) { n = F.a; fz = 0; }
    const int fl = n - F.a;
    if (fl < 0 || fl >= F.ns + 1) { key[ip] = (unsigned long long)nbin; return; }
    int ix = int(floor(wrap_mod(P.x[ip], F.Lx) / F.dx)), iy = int(floor(wrap_mod(P.y[ip], F.Ly) / F.dy));
    ix = ix < 0 ? 0 : (ix >= F.nx ? F.nx - 1 : ix);
    iy = iy < 0 ? 0 : (iy >= F.ny ? F.ny - 1 : iy);
    key[ip] = (unsigned long long)((long(fl) * nty + iy / kBT) * ntx + ix / kBT);
}
// the chunks of the bins: the head of each run of equal keys lists its run in chunks of at most kBChunk
__global__ void __launch_bounds__(kT) k_bpush_chunks(const unsigned long long* key, long n, long* chunk, int* nchunk,
                                                     int cap) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned long long k = key[i];
    if (k == kBNone || (i > 0 && key[i - 1] == k)) return;
    long lo = i + 1, hi = n;
    while (lo < hi) {
        const long mid = lo + ((hi - lo) >> 1);
        if (key[mid] == k) lo = mid + 1; else hi = mid;
    }
    const int m = int((lo - i + kBChunk - 1) / kBChunk);
    const int r = atomicAdd(nchunk, m);
    for (int q = 0; q < m && r + q < cap; ++q) {
        chunk[2 * (r + q)] = i + long(q) * kBChunk;
        chunk[2 * (r + q) + 1] = min(lo, i + long(q + 1) * kBChunk);
    }
}
// persistent: workgroup g takes the chunks g, g + grid, ...; every workgroup leaves when the list is done
__global__ void __launch_bounds__(kT) k_bunch_push_win(PushArgs c, Parts P, const unsigned long long* key,
                                                       const unsigned* idx, const long* chunk, const int* nchunk,
                                                       int cap, int ntx, int nty, long nbin, double z0) {
    __shared__ f4v win[3 * kBW * kBW];
    const FieldView& F = c.fv;
    const int nc = min(*nchunk, cap);
    for (int q = blockIdx.x; q < nc; q += gridDim.x) {
        const long lo = chunk[2 * q], hi = chunk[2 * q + 1];
        const unsigned long long k = key[lo];
        const int tx = int(k % (unsigned long long)ntx), ty = int((k / ntx) % (unsigned long long)nty);
        const int fl = int(k / ((unsigned long long)ntx * nty));
        const int x0 = tx * kBT - 1 - kBM, y0 = ty * kBT - 1 - kBM;
        constexpr int pl = kBW * kBW;
        const long cs = long(F.ns + 2) * F.nk;
        const bool none = k == (unsigned long long)nbin;   // outside the slices of F: no window (WX = 0)
        __syncthreads();                             // the previous chunk's particles are done with the window
        for (int r = none ? pl : threadIdx.x; r < pl; r += blockDim.x) {
            const int v = r / kBW, u = r - v * kBW;
            const float* src = F.F + long(fl) * F.nk + long(wrap_index(y0 + v, F.ny)) * F.nx + wrap_index(x0 + u, F.nx);
            win_node((G3D_LDS f4v*)win + 3 * r, src, cs, F.nk, true);
        }
        __syncthreads();
        const Win w{nullptr, (const G3D_LDS f4v*)win, nullptr, x0, y0, none ? 0 : kBW, kBW, fl, 0, 0};
        for (long t = lo + threadIdx.x; t < hi; t += blockDim.x) push_beam_one(c, w, P, long(idx[t]), z0);
    }
}

// TSC deposit of f (dt/Delta) v/(h dx dy) (src/sim_stream.hpp:33-64) into plane comp of the half-cell current:
// the tile's LDS window when the whole 3 x 3 stencil lies inside it, else jsr with global atomics.  Zero
// contributions are skipped (adding +-0 to a sum that starts at +0 never changes it).  The charge density planes
// only when rho: their one reader, the density lines, takes the last pass of a half-cell.
// a deposit into the current planes: float atomics in the FP32-mixed form (c.Jf), else FP64
__device__ __forceinline__ void jadd(const StreamArgs& c, long k, double v) {
    if (c.Jf) atomicAdd(&c.Jf[k], float(v));
    else atomicAdd(&c.J[k], v);
}

template <int YF>
__device__ __forceinline__ void sdeposit(const StreamArgs& c, const Win& win, double x, double y, double f, double vx,
                                         double vy, double vz, bool rho) {
    const FieldView& P = c.fv;
    int ix[3], jn[3], jh[3]; double wx[3], wn[3], wh[3];
    tsc_periodic(x, P.dx, P.nx, ix, wx);
    const long nk = P.nk;
    const int cq = f < 0 ? 3 : 4;
    const bool mv = vx != 0 || vy != 0 || vz != 0;
    if (YF == 1) {
        tsc_periodic(y, P.dy, P.ny, jn, wn);
        double w[9];
#pragma unroll
        for (int v = 0; v < 3; ++v)
#pragma unroll
            for (int u = 0; u < 3; ++u) w[3 * v + u] = f * wx[u] * wn[v] * c.ia[0];
        int u0 = 0, v0 = 0;
        bool in = false;
        if (win.WX) {
            u0 = wrap_index(ix[0] - win.x0, P.nx);
            v0 = wrap_index(jn[0] - win.y0, P.ny);
            in = u0 + 2 < win.WX && v0 + 2 < win.WY;
        }
        if (in) {
            const long wpl = long(win.WX) * win.WY;
#pragma unroll
            for (int v = 0; v < 3; ++v)
#pragma unroll
                for (int u = 0; u < 3; ++u) {
                    const ldsd L = win.lds + long(v0 + v) * win.WX + (u0 + u);
                    const double ww = w[3 * v + u];
                    if (mv) {
                        lds_add(L, ww * vx);
                        lds_add(L + wpl, ww * vy);
                        lds_add(L + 2 * wpl, ww * vz);
                    }
                    if (rho) lds_add(L + cq * wpl, ww);
                }
            return;
        }
#pragma unroll
        for (int v = 0; v < 3; ++v)
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                const long k = long(jn[v]) * P.nx + ix[u];
                const double ww = w[3 * v + u];
                if (mv) {
                    jadd(c, k, ww * vx);
                    jadd(c, nk + k, ww * vy);
                    jadd(c, 2 * nk + k, ww * vz);
                }
                if (rho) jadd(c, cq * nk + k, ww);
            }
        return;
    }
    tsc_freehand_w(P.yax, win, y, jn, wn, jh, wh);
    if (win.WX) {
        // the window's rows are node (and half-node) indices from y0, not wrapped: the walls bound the grid
        const int u0 = wrap_index(ix[0] - win.x0, P.nx), vn = jn[0] - win.y0, vh = jh[0] - win.y0;
        if (u0 + 2 < win.WX && vn >= 0 && vn + 2 < win.WY && vh >= 0 && vh + 2 < win.WY) {
            const long wpl = long(win.WX) * win.WY;
#pragma unroll
            for (int v = 0; v < 3; ++v) {
                const bool nod = jn[v] >= 1 && jn[v] <= P.ny - 1, hal = jh[v] >= 0 && jh[v] <= P.ny - 1;
#pragma unroll
                for (int u = 0; u < 3; ++u) {
                    if (nod) {
                        const ldsd L = win.lds + long(vn + v) * win.WX + (u0 + u);
                        const double w = f * wx[u] * wn[v] * c.ia[jn[v]];
                        if (mv) { lds_add(L, w * vx); lds_add(L + 2 * wpl, w * vz); }
                        if (rho) lds_add(L + cq * wpl, w);
                    }
                    if (hal && mv) {
                        const ldsd L = win.lds + long(vh + v) * win.WX + (u0 + u);
                        lds_add(L + wpl, f * wx[u] * wh[v] * c.id[jh[v]] * vy);
                    }
                }
            }
            return;
        }
    }
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        const bool nod = jn[v] >= 1 && jn[v] <= P.ny - 1, hal = jh[v] >= 0 && jh[v] <= P.ny - 1;
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            if (nod) {
                const long k = long(jn[v]) * P.nx + ix[u];
                const double w = f * wx[u] * wn[v] * c.ia[jn[v]];
                if (mv) { jadd(c, k, w * vx); jadd(c, 2 * nk + k, w * vz); }
                if (rho) jadd(c, cq * nk + k, w);
            }
            if (hal && mv) {
                const long k = long(jh[v]) * P.nx + ix[u];
                jadd(c, nk + k, f * wx[u] * wh[v] * c.id[jh[v]] * vy);
            }
        }
    }
}

// E, B at (x, y, zeta) (x, y wrapped as the grid wants): from the tile's field window when it holds the stencil,
// else from F; the values are the same either way.  two: also E at zeta1 and zeta0 (the ends of an ion's path, where
// the ionization rate is taken), from the same stencil
template <int YF, bool TWO>
__device__ __forceinline__ void gather_stream(const FieldView& P, const Win& win, double x, double y, double zeta,
                                              double E[3], double B[3], bool two, double zeta1, double zeta0,
                                              double E1[3], double E0[3]) {
    if (win.fld) {
        double g, f, g1 = 0, f1 = 0, g0 = 0, f0 = 0;
        WinStencil s;
        bool got = win_pair(P, win, zeta, g, f);
        if (TWO && two) got = got && win_pair(P, win, zeta1, g1, f1) && win_pair(P, win, zeta0, g0, f0);
        if (got && win_stencil<YF>(P, win, x, y, s)) {
            if (TWO && two) win_sums<YF, true>(win, s, g, f, E, B, g1, f1, g0, f0, E1, E0);
            else win_sums<YF, false>(win, s, g, f, E, B, 0, 0, 0, 0, nullptr, nullptr);
            return;
        }
    }
    if (TWO && two) {
        double D[3];
        gather_t<YF>(P, x, y, zeta1, E1, D);
        gather_t<YF>(P, x, y, zeta0, E0, D);
    }
    gather_t<YF>(P, x, y, zeta, E, B);
}

// |E| of the grid (E) and the analytic laser (src/sim_stream.hpp:67-74)
template <bool LASER>
__device__ __forceinline__ double field_abs(const StreamArgs& c, double x, double z, double zeta, double E[3]) {
    if (LASER) {
        double Ee[3], Be[3];
        c.laser.field(x + c.X0, z, z - (zeta - c.zc), Ee, Be);
        for (int k = 0; k < 3; ++k) E[k] += Ee[k];
    }
    return sqrt(E[0] * E[0] + E[1] * E[1] + E[2] * E[2]);
}

struct PState {
    double x, y, zeta, px, py, pz, w, z, q, qm;
    int alive, sp;
    unsigned long long id;
};

// Monte Carlo ADK (src/sim_stream.hpp:80-101): sequential levels with exponential waiting times; every event
// clones the ion as an electron into the born list
__device__ __forceinline__ void ionize(const StreamArgs& c, PState& p, double E1, double E0, double dt) {
    const IonDev I = c.ions[p.sp - SP_ION];
    if (!I.ionizing || (E1 < I.Emin && E0 < I.Emin)) return;
    const uint64_t base = key_particle(c.key, p.id);
    int Z = int(floor(p.q + 0.5));
    const int Z0 = Z;
    unsigned draw = 0;
    double tleft = dt;
    while (Z < I.Zmax) {
        const AdkLevel L = c.adk[I.off + Z];
        const double w = 0.5 * (adk_rate(L, E1) + adk_rate(L, E0));
        if (!(w > 0)) break;
        const double tw = -log(1.0 - uniform01(base + draw++)) / w;
        if (tw > tleft) break;
        tleft -= tw; ++Z;
        const int j = atomicAdd(c.bcnt, 1);
        if (j < c.bcap) {
            const Parts& b = c.born;
            b.x[j] = p.x; b.y[j] = p.y; b.zeta[j] = p.zeta; b.px[j] = p.px; b.py[j] = p.py; b.pz[j] = p.pz;
            b.w[j] = p.w; b.z[j] = p.z; b.q[j] = -1; b.qm[j] = -1; b.rem[j] = 0;
            b.alive[j] = 1; b.sp[j] = SP_FREED + (p.sp - SP_ION); b.id[j] = p.id;
        }
    }
    if (Z != Z0) { p.q = Z; p.qm = Z / I.mass; }
}

// one particle through half-cell n (src/sim_stream.hpp:104-171)
// YF: the grid (1 Fourier y, 0 free-hand y); ION: the list may hold ions; LASER: the deck has the analytic laser
// (without it the laser's field is zero and its evaluation would only cost registers)
template <int YF, bool ION, bool LASER>
__device__ __forceinline__ void stream_one(const StreamArgs& c, const Win& win, PState& p) {
    const int n = c.n;
    const double zn = c.zs[n], zn1 = c.zs[n + 1], h = zn1 - zn;
    if (p.alive == 6) {
        if (p.zeta > zn) p.alive = 1;
        else return;
    }
    if (p.alive != 1) return;
    const double hl = p.zeta >= zn1 - 1e-9 * h ? h : (p.zeta - zn > 0 ? p.zeta - zn : 0.0);
    const FieldView& P = c.fv;
    const bool ion = ION && is_ion(p.sp);
    const bool ionizing = ion && c.ions[p.sp - SP_ION].ionizing, fixed = ion && !c.ions[p.sp - SP_ION].mobile;
    const bool rho = !c.skip_state;
    double E1a = 0, E0a = 0;             // |E| at the ends of the path of an ionizing ion
    double E[3], B[3];
    const double zeta0 = p.zeta;
    const double g0 = sqrt(1 + p.px * p.px + p.py * p.py + p.pz * p.pz);
    const double omv0 = (1 + p.px * p.px + p.py * p.py) / (g0 * (g0 + p.pz));
    const double dt0 = hl / omv0;
    double xm = p.x, ym = p.y, zm = p.z;
    if (!fixed) {
        xm = p.x + 0.5 * dt0 * p.px / g0; ym = p.y + 0.5 * dt0 * p.py / g0;
        zm = p.z + 0.5 * dt0 * p.pz / g0;
    }
    const double zetam = p.zeta - 0.5 * hl;
    {
        double E1[3], E0[3];
        const double xg = wrap_mod(xm, P.Lx), yg = YF ? wrap_mod(ym, P.Ly) : ym;
        gather_stream<YF, ION>(P, win, xg, yg, zetam, E, B, ionizing, zeta0, zn, E1, E0);
        if (ION && ionizing) {
            E1a = field_abs<LASER>(c, xm, zm, zeta0, E1);
            E0a = field_abs<LASER>(c, xm, zm, zn, E0);
        }
    }
    if (fixed) {
        const double f = p.q * p.w * hl / (c.Delta * h * P.dx);
        if (f != 0) sdeposit<YF>(c, win, p.x, p.y, f, 0, 0, 0, rho);
        p.zeta = zn;
        if (ionizing) ionize(c, p, E1a, E0a, hl);
        return;
    }
    if (LASER) {
        double Ee[3], Be[3];
        c.laser.field(xm + c.X0, zm, zm - (zetam - c.zc), Ee, Be);
        for (int k = 0; k < 3; ++k) { E[k] += Ee[k]; B[k] += Be[k]; }
    }
    double ux = p.px, uy = p.py, uz = p.pz;
    boris(ux, uy, uz, E, B, p.qm, dt0);
    double g1 = sqrt(1 + ux * ux + uy * uy + uz * uz);
    double dt = 2 * hl / (omv0 + (1 + ux * ux + uy * uy) / (g1 * (g1 + uz)));
    ux = p.px; uy = p.py; uz = p.pz;
    boris(ux, uy, uz, E, B, p.qm, dt);
    g1 = sqrt(1 + ux * ux + uy * uy + uz * uz);
    double vx = 0.5 * (p.px / g0 + ux / g1), vy = 0.5 * (p.py / g0 + uy / g1), vz = 0.5 * (p.pz / g0 + uz / g1);
    double zeta_end = zn;
    bool trapped = false;
    if (p.z + vz * dt >= c.sTrap) {
        const double vzc = vz > 1e-3 ? vz : 1e-3;
        const double dtp = (c.sTrap - p.z) / vzc > 0 ? (c.sTrap - p.z) / vzc : 0.0;
        ux = p.px; uy = p.py; uz = p.pz;
        boris(ux, uy, uz, E, B, p.qm, dtp);
        g1 = sqrt(1 + ux * ux + uy * uy + uz * uz);
        vx = 0.5 * (p.px / g0 + ux / g1); vy = 0.5 * (p.py / g0 + uy / g1); vz = 0.5 * (p.pz / g0 + uz / g1);
        dt = dtp;
        zeta_end = p.zeta - (1 - vz) * dtp;
        trapped = true;
    }
    const double xo = p.x, yo = p.y;
    p.x += vx * dt; p.y += vy * dt;
    p.z = trapped ? c.s1 : p.z + vz * dt;
    p.px = ux; p.py = uy; p.pz = uz;
    p.zeta = zeta_end;
    const bool out = !YF && (p.y < c.ylo || p.y > c.yhi);
    // the streaming current, then for a trapped particle that joins the beam its beam current (one copy of the
    // deposit in the code)
    double f = p.q * p.w * dt / (c.Delta * h * P.dx);
    double xd = 0.5 * (xo + p.x), yd = 0.5 * (yo + p.y);
    const double vze = uz / g1;
    const bool join = trapped && !out && vze >= c.vz_beam;
#pragma unroll 1
    for (int d = 0;; ++d) {
        if (f != 0 || d) sdeposit<YF>(c, win, xd, yd, f, vx, vy, vz, rho);
        if (d || !join) break;
        xd = p.x; yd = p.y; f = p.q * p.w / (h * P.dx * vze); vx = ux / g1; vy = uy / g1; vz = vze;
    }
    if (out) { p.alive = 0; return; }
    if (ION && ionizing && !trapped) ionize(c, p, E1a, E0a, dt);
    if (trapped) p.alive = 5;
}

__device__ __forceinline__ PState load_pstate(const Parts& S, long i) {
    return PState{S.x[i], S.y[i], S.zeta[i], S.px[i], S.py[i], S.pz[i], S.w[i], S.z[i], S.q[i], S.qm[i], S.alive[i],
                  S.sp[i], S.id[i]};
}

// p: the state of list entry i (loaded by the caller); the pushed state goes to D[i]
template <int YF, bool ION, bool LASER>
__device__ __forceinline__ void stream_index(const StreamArgs& c, const Win& win, PState p, Parts D, long i) {
    stream_one<YF, ION, LASER>(c, win, p);
    if (c.skip_state) return;
    D.x[i] = p.x; D.y[i] = p.y; D.zeta[i] = p.zeta; D.px[i] = p.px; D.py[i] = p.py; D.pz[i] = p.pz;
    D.z[i] = p.z; D.q[i] = p.q; D.qm[i] = p.qm; D.alive[i] = p.alive;
}

// waves per SIMD that the register allocation of an instance must allow (0: the compiler's choice): 4 for the plain
// electron kernel (28 us at 256 x 256 against 31 with 3); the others spill too much for a cap (free-hand y with ions at
// 512 x 386: 439 us with 2 waves, 528 capped for 4)
constexpr int stream_waves(int YF, bool ION, bool LASER) { return YF == 1 && !ION && !LASER ? 4 : 1; }

// workgroups 0 .. ntile-1: the particles of one tile with the LDS window, added to the current planes at the end (or,
// without aflush, written to the tile's slab);
// the following workgroups: the untiled particles from off[ntile] on, one per lane, global atomics
// TILES: false for a list without tiles (the windows' code and registers left out).  Fourier y: a workgroup's deposits
// are summed in an LDS box around its particles' midpoints, where they fit one (a list in the order of its lattice); the
// deposits that miss the box, or find none, take the global atomics, 36 per particle, which bounded the kernel.  With the
// spectra of the current: 8.2 x 10^3 electrons at 2 per cell 31 -> 23 us, 3.3 x 10^4 at 2 per cell 49 -> 26, 2.0 x 10^5
// at 3 per cell 216 -> 52; 4.1 x 10^3 at 1 per cell 25 -> 23 (a chain of loads and FP64 operations of one wave, 15 us)
constexpr int kBoxNodes = 8;          // the largest box, per lane: 5 planes of 8 nodes, 20 KB for 64 lanes
template <int YF, bool ION, bool LASER, bool TILES>
__global__ void __launch_bounds__(kStreamBlockMax)
__attribute__((amdgpu_waves_per_eu(TILES ? stream_waves(YF, ION, LASER) : 1))) k_stream_halfcell(StreamArgs c, Parts S, Parts D, long n,
                                                                     TileGeom tg) {
    extern __shared__ __align__(16) double win_lds[];
    const long b = blockIdx.x;
    const bool tiled = TILES && b < tg.ntile;
    // free-hand y (every gather reads F): the tiles of one XCD a band of consecutive tile rows, so that
    // neighbouring tiles meet in one L2 (workgroup b runs on XCD b mod 8)
    const long t = (tg.fh && (tg.ntile & 7) == 0) ? (b & 7) * (tg.ntile >> 3) + (b >> 3) : b;
    // the particles binned into this tile (tg.idx: indices into the list; null: the contiguous load ranges), or a
    // block of the untiled rest.  The range, this lane's first particle and its state first: their dependent loads
    // overlap those of the field window.
    const int* idx = tiled ? tg.idx : nullptr;
    const long lo = tiled ? tg.off[t] : tg.n_tiled + (b - tg.ntile) * blockDim.x;
    const long hi = tiled ? tg.off[t + 1] : (lo + blockDim.x < n ? lo + blockDim.x : n);
    long k = lo + threadIdx.x;
    long i = k < hi ? (idx ? long(idx[k]) : k) : 0;
    PState p{};
    if (k < hi) p = load_pstate(S, i);
    const int pl = tg.WX * tg.WY;
    const long wn = 5L * pl;
    const int tx = int(t % (tiled ? tg.ntx : 1)), ty = tiled ? int(t / tg.ntx) : 0;
    const int x0 = tx * tg.TX - 1 - tg.M, y0 = ty * tg.TY - 1 - tg.M;
    const FieldView& F = c.fv;
    const int fl = c.n - F.a;
    const ldsd dep = (ldsd)win_lds;
    Win w{};
    if (tiled) {
        G3D_LDS f4v* fw = (G3D_LDS f4v*)(dep + ((wn + 1) & ~1L));
        for (long r = threadIdx.x; r < wn; r += blockDim.x) dep[r] = 0;
        const bool fwin = tg.fwin && F.self;
        // slices fl, fl + 1 of the 6 components, one node per lane, 12 loads.  Free-hand y: the rows beyond the walls
        // are never read (zero)
        if (fwin)
            for (int r = threadIdx.x; r < pl; r += blockDim.x) {
                const int v = r / tg.WX, u = r - v * tg.WX;
                const int gx = wrap_index(x0 + u, F.nx), gy = YF ? wrap_index(y0 + v, F.ny) : y0 + v;
                const bool in = YF || (gy >= 0 && gy < F.ny);
                const float* src = F.F + long(fl) * F.nk + long(in ? gy : 0) * F.nx + gx;
                win_node(fw + 3 * r, src, long(F.ns + 2) * F.nk, F.nk, in);
            }
        w = Win{dep, fwin ? fw : nullptr, nullptr, x0, y0, tg.WX, tg.WY, fl, 0, 0};
        if (YF == 0 && !F.yax.uniform && F.yax.n >= 3) {         // the y nodes of the window's rows
            const int nn = F.yax.n;
            w.y_lo = y0 < 0 ? 0 : (y0 > nn - 2 ? nn - 2 : y0);
            const int hi_r = y0 + tg.WY > nn - 1 ? nn - 1 : (y0 + tg.WY < w.y_lo + 1 ? w.y_lo + 1 : y0 + tg.WY);
            w.nyn = hi_r - w.y_lo;
            const ldsd hx = (ldsd)(fw + (fwin ? 3 * pl : 0));
            for (int r = threadIdx.x; r <= w.nyn; r += blockDim.x) hx[r] = F.yax.X[w.y_lo + r];
            w.yn = hx;
        }
        __syncthreads();
    }
    const double zn = c.zs[c.n];
    NodeBox box{};
    if (!TILES && YF == 1) {
        const bool on = k < hi && (p.alive == 1 || (p.alive == 6 && p.zeta > zn));
        const double h = c.zs[c.n + 1] - zn, g0 = sqrt(1 + p.px * p.px + p.py * p.py + p.pz * p.pz);
        const double t = 0.5 * (p.zeta - zn < h ? p.zeta - zn : h) * (g0 + p.pz) / (1 + p.px * p.px + p.py * p.py);
        box = node_box(on, mid_node(wrap_mod(p.x + t * p.px, F.Lx), F.dx, F.nx),
                       mid_node(wrap_mod(p.y + t * p.py, F.Ly), F.dy, F.ny), F.nx, F.ny, int(hi - lo), kBoxNodes * blockDim.x);
        for (int r = threadIdx.x; r < 5 * box.W * box.H; r += blockDim.x) dep[r] = 0;
        w = Win{dep, nullptr, nullptr, box.x0, box.y0, box.W, box.H, fl, 0, 0};
        __syncthreads();
    }
    unsigned cnt = 0;
    while (k < hi) {
        cnt += pushed_through(p.alive, p.zeta, zn);
        stream_index<YF, ION, LASER>(c, w, p, D, i);
        k += blockDim.x;
        if (k < hi) {
            i = idx ? long(idx[k]) : k;
            p = load_pstate(S, i);
        }
    }
    if (tiled) {
        __syncthreads();
        if (YF == 1 && !c.Jf && !tg.aflush) {
            double* sl = tg.slab + t * wn;
            for (long r = threadIdx.x; r < wn; r += blockDim.x) sl[r] = dep[r];
        } else                  // into the current planes (free-hand y: rows outside the walls hold nothing)
            for (long r = threadIdx.x; r < wn; r += blockDim.x) {
                const double v = dep[r];
                if (v == 0) continue;
                const int cc = int(r / pl), rr = int(r - long(cc) * pl), vv = rr / tg.WX, u = rr - vv * tg.WX;
                const int gy = YF ? wrap_index(y0 + vv, F.ny) : y0 + vv;
                if (gy < 0 || gy >= F.ny) continue;
                jadd(c, cc * F.nk + long(gy) * F.nx + wrap_index(x0 + u, F.nx), v);
            }
    }
    if (!TILES && YF == 1) {
        __syncthreads();
        const int nb = box.W * box.H;
        const float iw = 1.0f / float(box.W);
        for (int r = threadIdx.x; r < nb; r += blockDim.x) {
            double s[5];
#pragma unroll
            for (int cc = 0; cc < 5; ++cc) s[cc] = dep[cc * nb + r];
            const int q = box_node(box, iw, r, F.nx, F.ny);
#pragma unroll
            for (int cc = 0; cc < 5; ++cc)
                if (s[cc] != 0) jadd(c, cc * F.nk + q, s[cc]);
        }
    }
    if (c.npush) add_pushes(c.npush, cnt);
}

// ---------------------------------------------------------------- binning of the streaming list by tile
// The list keeps its order in memory; a tile's workgroup visits the particles whose current cell lies in the tile
// (idx[off[t] .. off[t+1])), so that particles that have moved away from their loading tile still deposit into
// and gather from LDS windows.  Only live particles (alive 1, waiting 6) are binned: the others are final for the
// rest of the step, and their state is copied into the second buffer here so that both buffers agree.
__device__ __forceinline__ int tile_of(const TileGeom& tg, double x, double y, double dx, double dy, int nx, int ny) {
    int ix = int(floor(x / dx)) % nx, iy;
    if (ix < 0) ix += nx;
    if (tg.fh) {                // free-hand y: the cell of the node table, clamped to the grid
        double f;
        tg.fy.locate(y, iy, f);
        iy = iy < 0 ? 0 : (iy >= ny ? ny - 1 : iy);
    } else {
        iy = int(floor(y / dy)) % ny;
        if (iy < 0) iy += ny;
    }
    return (iy / tg.TY) * tg.ntx + ix / tg.TX;
}
__global__ void __launch_bounds__(kT) k_bin_count(Parts S, Parts D, long n, TileGeom tg, double dx, double dy,
                                                  int nx, int ny, int* cnt) {
    extern __shared__ int hist[];
    for (int t = threadIdx.x; t < tg.ntile; t += blockDim.x) hist[t] = 0;
    __syncthreads();
    for (long i = long(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += long(gridDim.x) * blockDim.x) {
        const int al = S.alive[i];
        if (al == 1 || al == 6) atomicAdd(&hist[tile_of(tg, S.x[i], S.y[i], dx, dy, nx, ny)], 1);
        else {
            D.x[i] = S.x[i]; D.y[i] = S.y[i]; D.zeta[i] = S.zeta[i]; D.px[i] = S.px[i]; D.py[i] = S.py[i];
            D.pz[i] = S.pz[i]; D.z[i] = S.z[i]; D.q[i] = S.q[i]; D.qm[i] = S.qm[i]; D.alive[i] = al;
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < tg.ntile; t += blockDim.x)
        if (hist[t]) atomicAdd(&cnt[t], hist[t]);
}
// exclusive scan of the tile counts into off[0 .. ntile] and the scatter cursors (one workgroup: a chunk of tiles
// per lane, then a Hillis-Steele scan of the 1024 chunk sums)
__global__ void __launch_bounds__(1024) k_bin_scan(const int* cnt, long* off, int* cur, long ntile) {
    __shared__ long part[2][1024];
    const long per = (ntile + blockDim.x - 1) / blockDim.x;
    const long t0 = threadIdx.x * per, t1 = t0 + per < ntile ? t0 + per : ntile;
    long s = 0;
    for (long t = t0; t < t1; ++t) s += cnt[t];
    int src = 0;
    part[0][threadIdx.x] = s;
    __syncthreads();
    for (unsigned d = 1; d < blockDim.x; d <<= 1) {
        const long v = part[src][threadIdx.x] + (threadIdx.x >= d ? part[src][threadIdx.x - d] : 0);
        part[1 - src][threadIdx.x] = v;
        src = 1 - src;
        __syncthreads();
    }
    long a = part[src][threadIdx.x] - s;             // exclusive prefix of this lane's chunk
    for (long t = t0; t < t1; ++t) { off[t] = a; cur[t] = int(a); a += cnt[t]; }
    if (threadIdx.x == blockDim.x - 1) off[ntile] = part[src][threadIdx.x];
}
// one lane per particle: its rank among the workgroup's particles of the same tile (LDS atomics), one global
// reservation per tile the workgroup touches, then the index into its slot
__global__ void __launch_bounds__(kT) k_bin_scatter(Parts S, long n, TileGeom tg, double dx, double dy, int nx,
                                                    int ny, int* cur, int* idx) {
    extern __shared__ int lcnt[];                    // [ntile] counts, then [ntile] reserved bases
    int* lbase = lcnt + tg.ntile;
    for (int t = threadIdx.x; t < tg.ntile; t += blockDim.x) lcnt[t] = 0;
    __syncthreads();
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    int t = -1, r = 0;
    if (i < n) {
        const int al = S.alive[i];
        if (al == 1 || al == 6) {
            t = tile_of(tg, S.x[i], S.y[i], dx, dy, nx, ny);
            r = atomicAdd(&lcnt[t], 1);
        }
    }
    __syncthreads();
    for (int u = threadIdx.x; u < tg.ntile; u += blockDim.x)
        if (lcnt[u]) lbase[u] = atomicAdd(&cur[u], lcnt[u]);
    __syncthreads();
    if (t >= 0) idx[lbase[t] + r] = int(i);
}
__global__ void k_append_born(Parts b, const int* bcnt, Parts p0, Parts p1, long base, long cap) {
    const long cnt = *bcnt;
    // a few workgroups stride over the count (a grid for the whole capacity, up to Zmax times the ions, only exits)
    for (long i = long(blockIdx.x) * blockDim.x + threadIdx.x; i < cnt && base + i < cap;
         i += long(gridDim.x) * blockDim.x) {
        const long d = base + i;
        for (Parts* t : {&p0, &p1}) {
            t->x[d] = b.x[i]; t->y[d] = b.y[i]; t->zeta[d] = b.zeta[i]; t->px[d] = b.px[i]; t->py[d] = b.py[i];
            t->pz[d] = b.pz[i]; t->z[d] = b.z[i]; t->q[d] = b.q[i]; t->qm[d] = b.qm[i]; t->alive[d] = b.alive[i];
        }
        p0.w[d] = b.w[i]; p0.sp[d] = b.sp[i]; p0.id[d] = b.id[i]; p0.rem[d] = 0;
    }
}

// ---------------------------------------------------------------- list tools
__global__ void k_centroid_partial(Parts P, long np, double X0, double Y0, double* part) {
    __shared__ double s[3][kT];
    double a = 0, b = 0, w = 0;
    for (long i = long(blockIdx.x) * kT + threadIdx.x; i < np; i += long(gridDim.x) * kT) {
        if (P.alive[i] != 1 || !is_bunch(P.sp[i])) continue;
        a += P.w[i] * (P.x[i] + X0); b += P.w[i] * (P.y[i] + Y0); w += P.w[i];
    }
    s[0][threadIdx.x] = a; s[1][threadIdx.x] = b; s[2][threadIdx.x] = w;
    __syncthreads();
    for (int o = kT / 2; o > 0; o >>= 1) {
        if (int(threadIdx.x) < o)
            for (int k = 0; k < 3; ++k) s[k][threadIdx.x] += s[k][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) for (int k = 0; k < 3; ++k) part[3 * blockIdx.x + k] = s[k][0];
}
constexpr int kCentroidBlocks = 256;
// the partial sums staged in LDS by the whole workgroup, then added in block order by one lane (the loads off its
// chain of additions; the same sums in the same order)
__global__ void k_centroid_final(const double* part, int nb, double* out) {
    __shared__ double s[3 * kCentroidBlocks];
    for (int k = threadIdx.x; k < 3 * nb; k += blockDim.x) s[k] = part[k];
    __syncthreads();
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double a = 0, b = 0, w = 0;
    for (int k = 0; k < nb; ++k) { a += s[3 * k]; b += s[3 * k + 1]; w += s[3 * k + 2]; }
    out[0] = a; out[1] = b; out[2] = w;
}

__device__ void to_aos(const Parts& p, long i, g3d_particle& o) {
    o.x = p.x[i]; o.y = p.y[i]; o.zeta = p.zeta[i]; o.px = p.px[i]; o.py = p.py[i]; o.pz = p.pz[i]; o.w = p.w[i];
    o.rem = p.rem[i]; o.z = p.z[i]; o.q = p.q[i]; o.qm = p.qm[i]; o.alive = p.alive[i]; o.sp = p.sp[i]; o.id = p.id[i];
}
__global__ void k_collect(Parts p, long n, int code, g3d_particle* out, long* idx, int* count, long cap) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n || p.alive[i] != code) return;
    const int j = atomicAdd(count, 1);
    if (j >= cap) return;
    to_aos(p, i, out[j]);
    idx[j] = i;
}
__global__ void k_count(Parts p, long n, int code, int* count) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    const bool hit = i < n && p.alive[i] == code;
    const unsigned long long m = __ballot(hit);
    if (m && (threadIdx.x & 63) == 0) atomicAdd(count, int(__popcll(m)));
}
__global__ void k_from_aos(const g3d_particle* in, Parts p, long n) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const g3d_particle o = in[i];
    p.x[i] = o.x; p.y[i] = o.y; p.zeta[i] = o.zeta; p.px[i] = o.px; p.py[i] = o.py; p.pz[i] = o.pz; p.w[i] = o.w;
    p.rem[i] = o.rem; p.z[i] = o.z; p.q[i] = o.q; p.qm[i] = o.qm; p.alive[i] = o.alive; p.sp[i] = o.sp; p.id[i] = o.id;
}
__global__ void k_to_aos(Parts p, g3d_particle* out, long n) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    to_aos(p, i, out[i]);
}
__global__ void k_copy(Parts s, Parts d, long n) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    d.x[i] = s.x[i]; d.y[i] = s.y[i]; d.zeta[i] = s.zeta[i]; d.px[i] = s.px[i]; d.py[i] = s.py[i]; d.pz[i] = s.pz[i];
    d.z[i] = s.z[i]; d.q[i] = s.q[i]; d.qm[i] = s.qm[i]; d.alive[i] = s.alive[i];
}
__global__ void k_shift(Parts p, long n, double sx, double sy) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    p.x[i] -= sx; p.y[i] -= sy;
}
}  // namespace

void bunch_push(const PushArgs& a, Parts p, long np, double s0) {
    if (np <= 0) return;
    hipLaunchKernelGGL(k_bunch_push, dim3(blocks_for(np, kT)), dim3(kT), 0, stream(), a, p, np, s0);
    launch_check("bunch push");
}
void bunch_push_windowed(const PushArgs& a, Parts p, long np, double s0, BpushScratch& s) {
    if (np <= 0) return;
    const FieldView& F = a.fv;
    if (!F.yf || !F.self || F.nx < 2 * kBT || F.ny < 2 * kBT || np > long(0xffffffffu)) {
        bunch_push(a, p, np, s0);
        return;
    }
    const int ntx = (F.nx + kBT - 1) / kBT, nty = (F.ny + kBT - 1) / kBT;
    const long nbin = long(F.ns + 1) * nty * ntx;
    int eb = 1;                                      // bits of the bins and the bin nbin, one more for ~0
    while ((1ll << eb) <= nbin) ++eb;
    ++eb;
    if (s.key0.size() < size_t(np)) {
        const size_t cap = size_t(np) + size_t(np) / 4;
        s.key0.resize(cap); s.key1.resize(cap); s.idx0.resize(cap); s.idx1.resize(cap);
    }
    const int cap = int(np / 1 + 1);                 // chunks: at most one per particle
    if (s.chunk.size() < size_t(2 * cap)) s.chunk.resize(size_t(2 * cap));
    if (s.nchunk.size() < 1) s.nchunk.resize(1);
    hipLaunchKernelGGL(k_bpush_keys, dim3(blocks_for(np, kT)), dim3(kT), 0, stream(), a, p, np, ntx, nty, nbin,
                       s.key0.data(), s.idx0.data());
    auto sort = [&](auto config) {
        size_t bytes = 0;
        hip_check(rocprim::radix_sort_pairs<decltype(config)>(nullptr, bytes, s.key0.data(), s.key1.data(), s.idx0.data(),
                                                              s.idx1.data(), np, 0, unsigned(eb), stream()), "beam push sort size");
        if (s.tmp.size() < bytes) s.tmp.resize(bytes + bytes / 4 + 256);
        bytes = s.tmp.size();
        hip_check(rocprim::radix_sort_pairs<decltype(config)>(s.tmp.data(), bytes, s.key0.data(), s.key1.data(), s.idx0.data(),
                                                              s.idx1.data(), np, 0, unsigned(eb), stream()), "beam push sort");
    };
    if (np <= kBpushMerge) sort(rocprim::default_config{});
    else sort(BpushSort{});
    hip_check(hipMemsetAsync(s.nchunk.data(), 0, sizeof(int), stream()), "hipMemsetAsync");
    hipLaunchKernelGGL(k_bpush_chunks, dim3(blocks_for(np, kT)), dim3(kT), 0, stream(), s.key1.data(), np,
                       s.chunk.data(), s.nchunk.data(), cap);
    hipLaunchKernelGGL(k_bunch_push_win, dim3(2048), dim3(kT), 0, stream(), a, p, s.key1.data(), s.idx1.data(),
                       s.chunk.data(), s.nchunk.data(), cap, ntx, nty, nbin, s0);
    launch_check("bunch push (windows)");
}
void stream_halfcell(const StreamArgs& a, Parts src, Parts dst, long nstrm, const TileGeom& tg,
                     const LaunchTimer& lt) {
    if (nstrm <= 0) return;
    // tile workgroups of tg.block lanes, then the untiled tail in workgroups of the same size
    // (an untiled list in workgroups of one wave: Fourier y, 128 lanes are 1 to 4 us slower where the list has a part in
    // no order, whose atomics the few waves of a larger workgroup hide less, and at most 2 us faster elsewhere; free-hand
    // y, a short list's few waves then spread over the compute units)
    const int bs = tg.ntile ? tg.block : (a.fv.yf || nstrm <= 6144 ? 64 : kT);
    if (bs < 64 || bs > kStreamBlockMax || bs % 64) throw std::runtime_error("stream half-cell: bad block size");
    const long tail_blocks = nstrm > tg.n_tiled ? long(blocks_for(nstrm - tg.n_tiled, bs)) : 0;
    // the deposit window (5 double planes, an even number of values), the field window (12 floats per node) and the
    // window's y nodes of the free-hand grid
    const size_t pl = size_t(tg.WX) * tg.WY;
    const size_t lds = tg.ntile ? ((5 * pl + 1) & ~size_t(1)) * sizeof(double) + (tg.fwin ? pl * 12 * sizeof(float) : 0) +
                                      (a.fv.yf ? 0 : size_t(tg.WY + 2) * sizeof(double))
                                : (a.fv.yf ? size_t(5) * kBoxNodes * bs * sizeof(double) : 0);
    const dim3 grid(unsigned(tg.ntile + tail_blocks)), blk(bs);
    if (a.npush && long(grid.x) > a.npush_cap) throw std::runtime_error("stream half-cell: push counter too small");
    const bool ion = a.ions != nullptr;
    const unsigned sh = unsigned(lds);
    auto pick = [&](auto tiles) {
        constexpr bool T = decltype(tiles)::value;
        return a.laser.on
            ? (a.fv.yf ? (ion ? k_stream_halfcell<1, true, true, T> : k_stream_halfcell<1, false, true, T>)
                       : (ion ? k_stream_halfcell<0, true, true, T> : k_stream_halfcell<0, false, true, T>))
            : (a.fv.yf ? (ion ? k_stream_halfcell<1, true, false, T> : k_stream_halfcell<1, false, false, T>)
                       : (ion ? k_stream_halfcell<0, true, false, T> : k_stream_halfcell<0, false, false, T>));
    };
    auto* k = tg.ntile ? pick(std::true_type{}) : pick(std::false_type{});
    launch_timed_kernel(lt, k, grid, blk, sh, a, src, dst, nstrm, tg);
    launch_check("stream half-cell");
}
// one workgroup: the further chunks of every tile, listed through an LDS counter
__global__ void __launch_bounds__(1024) k_tile_chunks(const long* off, long ntile, int chunk, int cap, int* xtile,
                                                      long* xstart, int* xcount) {
    __shared__ int cnt;
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    for (long t = threadIdx.x; t < ntile; t += blockDim.x)
        for (long s = off[t] + chunk; s < off[t + 1]; s += chunk) {
            const int e = atomicAdd(&cnt, 1);
            if (e < cap) { xtile[e] = int(t); xstart[e] = s; }
        }
    __syncthreads();
    if (threadIdx.x == 0) xcount[0] = cnt < cap ? cnt : cap;
}
void tile_chunks(const TileGeom& tg, int* xtile, long* xstart, int* xcount) {
    if (tg.ntile <= 0 || tg.chunk <= 0) return;
    hipLaunchKernelGGL(k_tile_chunks, dim3(1), dim3(1024), 0, stream(), tg.off, tg.ntile, tg.chunk, tg.max_extra,
                       xtile, xstart, xcount);
    launch_check("tile chunks");
}
bool tile_shape(TileGeom& tg, int nx, int ny, bool yf, int M, int px, int py) {
    auto pick = [](int n, int pref) { for (int t = pref; t >= 8; t >>= 1) if (n % t == 0 && n >= 2 * t) return t; return 0; };
    if (!px || !py) { px = long(nx) * ny < 256L * 16 * 8 && yf ? 8 : 16; py = 8; }
    // free-hand y: rows of py cells from the first node (the last row may be short), the windows end at the walls
    const int TX = pick(nx, px), TY = yf ? pick(ny, py) : (ny >= 2 * py ? py : 0);
    if (!TX || !TY) return false;
    M = std::min({M, TX - 1, TY - 1, (nx - TX - 3) / 2});
    if (yf) M = std::min(M, (ny - TY - 3) / 2);
    if (M < 0) return false;
    tg.TX = TX; tg.TY = TY; tg.M = M; tg.WX = TX + 3 + 2 * M; tg.WY = TY + 3 + 2 * M;
    tg.ntx = nx / TX; tg.nty = (ny + TY - 1) / TY; tg.ntile = long(tg.ntx) * tg.nty;
    return true;
}
void bin_tiles(Parts S, Parts D, long n, const TileGeom& tg, double dx, double dy, int nx, int ny, int* cnt,
               int* cur, long* off, int* idx) {
    if (n <= 0 || tg.ntile <= 0) return;
    if (tg.ntile > 16384) throw std::runtime_error("bin tiles: more than 16384 tiles");
    hip_check(hipMemsetAsync(cnt, 0, sizeof(int) * size_t(tg.ntile), stream()), "hipMemsetAsync");
    const unsigned blocks = unsigned(std::min<long>(1024, long(blocks_for(n, kT))));
    hipLaunchKernelGGL(k_bin_count, dim3(blocks), dim3(kT), sizeof(int) * size_t(tg.ntile), stream(), S, D, n, tg, dx,
                       dy, nx, ny, cnt);
    hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(1024), 0, stream(), cnt, off, cur, tg.ntile);
    hipLaunchKernelGGL(k_bin_scatter, dim3(blocks_for(n, kT)), dim3(kT), 2 * sizeof(int) * size_t(tg.ntile), stream(),
                       S, n, tg, dx, dy, nx, ny, cur, idx);
    launch_check("bin tiles");
}
void append_born(Parts born, const int* bcnt, Parts p0, Parts p1, long base, long cap) {
    if (cap <= base) return;
    const unsigned nb = std::min(blocks_for(cap - base, kT), 128u);
    hipLaunchKernelGGL(k_append_born, dim3(nb), dim3(kT), 0, stream(), born, bcnt, p0, p1, base, cap);
    launch_check("append born");
}
void bunch_centroid(Parts p, long np, double X0, double Y0, double* out3) {
    static double* part = nullptr;
    const int nb = kCentroidBlocks;
    if (!part) hip_check(hipMalloc(reinterpret_cast<void**>(&part), 3 * nb * sizeof(double)), "hipMalloc");
    hipLaunchKernelGGL(k_centroid_partial, dim3(nb), dim3(kT), 0, stream(), p, np, X0, Y0, part);
    hipLaunchKernelGGL(k_centroid_final, dim3(1), dim3(64), 0, stream(), part, nb, out3);
    launch_check("centroid");
}
void collect_alive(Parts p, long n, int code, g3d_particle* out, long* idx, int* count, long cap) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_collect, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), p, n, code, out, idx, count, cap);
    launch_check("collect");
}
void count_alive(Parts p, long n, int code, int* count) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_count, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), p, n, code, count);
    launch_check("count");
}
void parts_from_aos(const g3d_particle* in, Parts p, long n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_from_aos, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), in, p, n);
    launch_check("particles from AoS");
}
void parts_to_aos(Parts p, g3d_particle* out, long n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_to_aos, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), p, out, n);
    launch_check("particles to AoS");
}
// the fresh plasma lattice of a step, generated in tile order (see LatticeArgs), one workgroup per tile; both list
// buffers
__global__ void __launch_bounds__(kT) k_lattice(LatticeArgs L, Parts A, Parts B) {
    const long t = blockIdx.x;
    const int tx = int(t % L.ntx), ty = int(t / L.ntx);
    const int jt = ty * L.TY, ja = jt < L.j0 ? L.j0 : jt;      // the tile's first loaded row
    const long lo = L.off[t], n = L.off[t + 1] - lo;
    const int pp = L.px * L.py;
    const int per = int(n / (L.nsp * pp));                     // cells of the tile
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
        const int k = r / (pp * per), rk = r - k * pp * per;
        const int sub = rk / per, c = rk - sub * per;
        const int jl = c / L.TX, il = c - jl * L.TX;
        const int b2 = sub / L.px, a2 = sub - b2 * L.px;
        const int j = ja + jl, i = tx * L.TX + il;
        // the host loader's formulas and operation order (src/sim_plasma.cpp:62-64)
        const double y0 = L.yn ? L.yn[j] : j * L.dy, hy = L.yn ? L.yn[j + 1] - L.yn[j] : L.dy;
        const double x = (i + (a2 + 0.5) / L.px) * L.dx;
        const double y = y0 + (b2 + 0.5) / L.py * hy;
        const double X = x + L.X0, Y = y + L.Y0, r2 = X * X + Y * Y;
        const double gch = L.parabolic ? 1 + L.channel_depth * r2 / (L.r_channel * L.r_channel) : 1.0;
        const double dens = L.f * gch > 0 ? L.n0 * L.f * gch : 0.0;
        const LatticeSpecies S = L.sp[k];
        const double w = S.atoms * (dens * L.dx * hy * L.Delta / (L.px * L.py));
        const long g = lo + r;
        A.x[g] = x; A.y[g] = y; A.zeta[g] = L.zf; A.px[g] = 0; A.py[g] = 0; A.pz[g] = 0; A.w[g] = w; A.rem[g] = 0;
        A.z[g] = L.s0; A.q[g] = S.q; A.qm[g] = S.qm; A.alive[g] = 1; A.sp[g] = S.sp;
        A.id[g] = L.id0 + ((((unsigned long long)(j - L.j0) * L.nx + i) * L.py + b2) * L.px + a2) * L.nsp + k;
        B.x[g] = x; B.y[g] = y; B.zeta[g] = L.zf; B.px[g] = 0; B.py[g] = 0; B.pz[g] = 0; B.z[g] = L.s0; B.q[g] = S.q;
        B.qm[g] = S.qm; B.alive[g] = 1;
    }
}
void plasma_lattice(const LatticeArgs& L, Parts A, Parts B, long ntile) {
    if (ntile <= 0) return;
    hipLaunchKernelGGL(k_lattice, dim3(unsigned(ntile)), dim3(kT), 0, stream(), L, A, B);
    launch_check("plasma lattice");
}

// ion statistics: every lane its own sums in LDS ([slot][lane]), then a tree over the lanes of the workgroup, then
// the workgroups in order
constexpr int kIonStatLanes = 64;
__global__ void __launch_bounds__(kIonStatLanes) k_ion_stats(IonStatArgs a, Parts p, long n, double* part) {
    extern __shared__ double ist[];
    const int t = threadIdx.x;
    for (int s = 0; s < a.nslot; ++s) ist[s * kIonStatLanes + t] = 0;
    for (long i = long(blockIdx.x) * kIonStatLanes + t; i < n; i += long(gridDim.x) * kIonStatLanes) {
        const int sp = p.sp[i];
        if (sp < SP_ION || sp >= SP_ION + 4) continue;
        const IonStatSpecies S = a.s[sp - SP_ION];
        if (S.slot < 0) continue;
        const int Z = int(floor(p.q[i] + 0.5));
        const double w = p.w[i];
        if (p.alive[i] == 1 && Z >= 0 && Z <= S.Zmax) ist[(S.slot + Z) * kIonStatLanes + t] += w;
        ist[(S.slot + S.Zmax + 1) * kIonStatLanes + t] += (Z - S.Z0) * w;
        ist[(S.slot + S.Zmax + 2) * kIonStatLanes + t] += 1;
    }
    __syncthreads();
    for (int o = kIonStatLanes / 2; o > 0; o >>= 1) {
        if (t < o)
            for (int s = 0; s < a.nslot; ++s) ist[s * kIonStatLanes + t] += ist[s * kIonStatLanes + t + o];
        __syncthreads();
    }
    for (int s = t; s < a.nslot; s += kIonStatLanes) part[long(blockIdx.x) * a.nslot + s] = ist[s * kIonStatLanes];
}
__global__ void k_ion_stats_final(const double* part, int nslot, int nb, double* out) {
    const int s = threadIdx.x;
    if (s >= nslot) return;
    double v = 0;
    for (int b = 0; b < nb; ++b) v += part[long(b) * nslot + s];
    out[s] = v;
}
void ion_statistics(const IonStatArgs& a, Parts p, long n, double* part, double* out) {
    if (a.nslot <= 0) return;
    if (a.nslot > 128) throw std::runtime_error("ion statistics: too many charge states");
    const size_t lds = size_t(a.nslot) * kIonStatLanes * sizeof(double);
    hipLaunchKernelGGL(k_ion_stats, dim3(kIonStatBlocks), dim3(kIonStatLanes), lds, stream(), a, p, n, part);
    hipLaunchKernelGGL(k_ion_stats_final, dim3(1), dim3(128), 0, stream(), part, a.nslot, kIonStatBlocks, out);
    launch_check("ion statistics");
}
void parts_copy(Parts s, Parts d, long n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_copy, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), s, d, n);
    launch_check("particles copy");
}
void parts_shift(Parts p, long n, double sx, double sy) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_shift, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), p, n, sx, sy);
    launch_check("particles shift");
}

}  // namespace g3d
