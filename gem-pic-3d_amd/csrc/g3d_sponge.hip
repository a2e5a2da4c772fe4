// The sponge and the real fields of all slices on the Fourier-y grid (src/sim_fields.cpp:156-307), and the spectra of
// the beam currents (src/sim_particles.cpp:120-158), each pointwise step fused into the transform next to it.
//
// Sponge (per slice):
//   1. k_sp_rows     the bound field psi of the beam, R - R_b packed, inverse transforms along the contiguous direction
//   2. k_sp_cols     inverse transforms across it, the masks of the sponge layers in real space, forward transforms
//                    back across (one LDS round trip for both)
//   3. k_sp_unpack   forward transforms along it; the packed pair unpacked with the mirrored row (both rows in one
//                    workgroup) and R_b added back: R_x, R_y
// Real fields:
//   4. k_pack_cols   the planes R_x + i R_y, L_x + i L_y, E_z + i B_z packed and y-transformed
//   5. k_rows_F      x transforms of the three planes of a row and E, B into the float F
// Every kernel moves each of its planes once: with psi 344 bytes per point (step 5's F and the inputs and outputs of the
// call are 168 of them) where separate pack, transform, mask and unpack kernels moved about 800; 256 x 256 x 256 points 2.32 -> 1.52 ms (1.85 TB/s of the 168 bytes; the copy rate is 5.1).
//
// The modes may be row-major (j nx + ix) or column-major (ix ny + j): steps 1-3 run the same code with the
// directions exchanged, step 4 reads either and writes row-major.  The order of the two directions differs from the
// batched transform's (rows then columns), so the results agree with it to rounding.
#include <algorithm>

#include "g3d_fft_core.hpp"
#include "g3d_kernels.hpp"
#include "g3d_runtime.hpp"

namespace g3d {
namespace {
using namespace fftcore;
constexpr int kT = 256;
constexpr int kTile = 2048;          // complex values per workgroup

__device__ __forceinline__ void unpack_pair(cx z, cx zm, cx& X, cx& Y) {
    X = 0.5 * (z + zm);
    const cx d = z - zm;
    Y = 0.5 * mk(d.im, -d.re);
}

// planes of n1 rows of n0 contiguous points; swap: the contiguous direction is y (column-major modes)
struct SpongeView {
    int n0, n1, l0, l1, ns, N, a, swap;
    long nk;
    const double *k0, *k1;           // k along and across the rows
    const double *hc, *wl, *wu;
    double g2, opb;
    const cx *jz, *tw0, *tw1;
    cx *rx, *ry, *s1, *s2;
};

// ---------------------------------------------------------------- 1
__global__ void __launch_bounds__(kT) k_sp_rows(SpongeView c, int rpw) {
    extern __shared__ __align__(16) unsigned char smraw[];
    cx* buf = reinterpret_cast<cx*>(smraw);
    const int n0 = c.n0, sp = padded(n0);
    cx* tws = buf + size_t(rpw) * sp;
    load_twiddles(tws, c.tw0, n0 >> 1, true);
    const long row0 = long(blockIdx.x) * rpw, left = (long(c.ns) << c.l1) - row0;
    const int nr = left < rpw ? int(left) : rpw, tot = nr << c.l0;
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> c.l0, i = e & (n0 - 1);
        const long row = row0 + r;
        const int l = int(row >> c.l1), j = int(row & (c.n1 - 1)), n = c.a + l;
        const long ic = (long(j) << c.l0) + i, idx = long(l) * c.nk + ic;
        // charge of slice n + dl from the filtered half-cell currents (the ghost half-cells of one GPU are zero)
        cx q[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const int p = l - 1 + h;
            q[h] = (p < 0 || p > c.ns) ? mk(0) : c.jz[long(p) * c.nk + ic];
        }
        auto rho_at = [&](int dl) -> cx {
            const int nn = n + dl;
            if (nn < 0 || nn > c.N - 1) return mk(0);
            return c.wl[nn] * q[dl + 1] + c.wu[nn] * q[dl + 2];
        };
        const double hm = c.hc[n + 1], hp = c.hc[n + 2];
        const double cm = 2 / ((hm + hp) * hm), cp = 2 / ((hm + hp) * hp);
        const double ka = c.k0[i], kb = c.k1[j], kxv = c.swap ? kb : ka, kyv = c.swap ? ka : kb;
        const double k2 = kxv * kxv + kyv * kyv;
        cx psi = mk(0);
        if (k2 > 0) {
            const cx r0 = rho_at(0);
            const cx d2 = c.g2 * (cp * rho_at(1) - (cm + cp) * r0 + cm * rho_at(-1));
            psi = (r0 + d2 / k2) / k2;
        }
        c.s2[idx] = psi;
        const cx bx = -c.opb * (ik(kxv) * psi), by = -c.opb * (ik(kyv) * psi);
        const cx u = c.rx[idx] - bx, v = c.ry[idx] - by;
        buf[r * sp + lpos(bitrev(i, c.l0))] = mk(u.re - v.im, u.im + v.re);
    }
    __syncthreads();
    lds_fft(buf, n0, c.l0, nr, sp, tws);
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> c.l0, i = e & (n0 - 1);
        c.s1[(row0 << c.l0) + e] = buf[r * sp + lpos(i)];
    }
}

// ---------------------------------------------------------------- 2
// ma: the mask along the rows, mre and mim across them (of the real and the imaginary part); scale: 1 / (nx ny)
__global__ void __launch_bounds__(kT) k_sp_cols(SpongeView c, int lnc, const double* mx, const double* mn,
                                                const double* mh, double scale) {
    extern __shared__ __align__(16) unsigned char smraw[];
    cx* buf = reinterpret_cast<cx*>(smraw);
    const int n1 = c.n1, sp = padded(n1), nc = 1 << lnc;
    cx* twi = buf + size_t(nc) * sp;
    cx* twf = twi + (n1 >> 1);
    load_twiddles(twi, c.tw1, n1 >> 1, true);
    load_twiddles(twf, c.tw1, n1 >> 1, false);
    const int tiles = c.n0 >> lnc;
    const long p = blockIdx.x / tiles;
    const int c0 = int(blockIdx.x - p * tiles) << lnc, tot = nc * n1;
    cx* g = c.s1 + p * c.nk + c0;
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int j = e >> lnc, q = e & (nc - 1);
        buf[q * sp + lpos(bitrev(j, c.l1))] = g[(long(j) << c.l0) + q];
    }
    __syncthreads();
    lds_fft(buf, n1, c.l1, nc, sp, twi);
    auto masked = [&](cx v, int j, int i) {
        v = scale * v;
        const int x = c.swap ? j : i, y = c.swap ? i : j;
        return mk(mx[x] * mn[y] * v.re, mx[x] * mh[y] * v.im);
    };
    // in place into the bit-reversed order of the forward transform: the pair (j, bitrev j) by one lane
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int q = e >> c.l1, j = e & (n1 - 1), b = bitrev(j, c.l1);
        if (b < j) continue;
        cx* s = buf + q * sp;
        const cx v = masked(s[lpos(j)], j, c0 + q);
        if (b != j) s[lpos(j)] = masked(s[lpos(b)], b, c0 + q);
        s[lpos(b)] = v;
    }
    __syncthreads();
    lds_fft(buf, n1, c.l1, nc, sp, twf);
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int j = e >> lnc, q = e & (nc - 1);
        g[(long(j) << c.l0) + q] = buf[q * sp + lpos(j)];
    }
}

// ---------------------------------------------------------------- 3
// pair m of a plane: rows m and n1 - m, each the other's mirror (m = 0: rows 0 and n1/2, each its own)
__global__ void __launch_bounds__(kT) k_sp_unpack(SpongeView c, int lpw) {
    extern __shared__ __align__(16) unsigned char smraw[];
    cx* buf = reinterpret_cast<cx*>(smraw);
    const int n0 = c.n0, sp = padded(n0), pw = 1 << lpw;
    cx* tws = buf + size_t(2 * pw) * sp;
    load_twiddles(tws, c.tw0, n0 >> 1, false);
    const int lh = c.l1 - 1;                          // pairs per plane: n1 / 2
    const long pair0 = long(blockIdx.x) << lpw;
    const int tot = 2 << (lpw + c.l0);
    auto row_of = [&](int r) -> long {                // sequence r: pair r / 2, its first or second row
        const long pr = pair0 + (r >> 1), l = pr >> lh;
        const int m = int(pr & ((1 << lh) - 1));
        return (l << c.l1) + ((r & 1) ? (m ? c.n1 - m : c.n1 >> 1) : m);
    };
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> c.l0, i = e & (n0 - 1);
        buf[r * sp + lpos(bitrev(i, c.l0))] = c.s1[(row_of(r) << c.l0) + i];
    }
    __syncthreads();
    lds_fft(buf, n0, c.l0, 2 * pw, sp, tws);
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> c.l0, i = e & (n0 - 1);
        const long row = row_of(r), idx = (row << c.l0) + i;
        const int j = int(row & (c.n1 - 1));
        const int rm = ((pair0 + (r >> 1)) & ((1 << lh) - 1)) ? (r ^ 1) : r;
        cx X, Y;
        unpack_pair(buf[r * sp + lpos(i)], conjg(buf[rm * sp + lpos((n0 - i) & (n0 - 1))]), X, Y);
        const double ka = c.k0[i], kb = c.k1[j], kxv = c.swap ? kb : ka, kyv = c.swap ? ka : kb;
        const cx psi = c.s2[idx];
        c.rx[idx] = X - c.opb * (ik(kxv) * psi);
        c.ry[idx] = Y - c.opb * (ik(kyv) * psi);
    }
}

// ---------------------------------------------------------------- 4
__device__ __forceinline__ void put(cx& d, cx v) { d = v; }
__device__ __forceinline__ void put(cxf& d, cx v) { d = to_f(v); }
struct PackView {
    const cx *a[3], *b[3];           // the pairs a + i b: R, L, (E_z, B_z)
    int nx, ny, lx, ly, cm;
    long nk;
};
// C: cx, or cxf for the FP32 transforms of the FP32-mixed form.  Workgroup: nc columns of one of the three planes
template <class C>
__global__ void __launch_bounds__(kT) k_pack_cols(PackView c, C* T, long ts, int lnc, long per, const cx* twy) {
    extern __shared__ __align__(16) unsigned char smraw[];
    C* buf = reinterpret_cast<C*>(smraw);
    const int ny = c.ny, sp = padded(ny), nc = 1 << lnc;
    C* tws = buf + size_t(nc) * sp;
    load_twiddles(tws, twy, ny >> 1, true);
    const int k = int(blockIdx.x / per);
    const long w = blockIdx.x - k * per;
    const int tiles = c.nx >> lnc;
    const long p = w / tiles;
    const int c0 = int(w - p * tiles) << lnc, tot = nc * ny;
    const cx* A = c.a[k] + p * c.nk;
    const cx* B = c.b[k] + p * c.nk;
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int j = c.cm ? e & (ny - 1) : e >> lnc, q = c.cm ? e >> c.ly : e & (nc - 1);
        const long i = c.cm ? (long(c0 + q) << c.ly) + j : (long(j) << c.lx) + c0 + q;
        const cx u = A[i], v = B[i];
        put(buf[q * sp + lpos(bitrev(j, c.ly))], mk(u.re - v.im, u.im + v.re));
    }
    __syncthreads();
    lds_fft(buf, ny, c.ly, nc, sp, tws);
    C* t = T + k * ts + p * c.nk + c0;
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int j = e >> lnc, q = e & (nc - 1);
        t[(long(j) << c.lx) + q] = buf[q * sp + lpos(j)];
    }
}

// ---------------------------------------------------------------- 5
// rows row0 ... of the planes of T; E_x = (R_x + L_x)/2, E_y = (R_y + L_y)/2, B_x = (L_y - R_y)/2, B_y = (R_x - L_x)/2
// (src/sim_fields.cpp:280-293), E_z, B_z into float F
template <class C, class S>
__global__ void __launch_bounds__(kT) k_rows_F(const C* T, long ts, float* F, long fpl, int nx, int lx, long nrows,
                                               int rpw, const cx* twx, S scale) {
    extern __shared__ __align__(16) unsigned char smraw[];
    C* buf = reinterpret_cast<C*>(smraw);
    const int sp = padded(nx);
    C* tws = buf + size_t(3 * rpw) * sp;
    load_twiddles(tws, twx, nx >> 1, true);
    const long row0 = long(blockIdx.x) * rpw, left = nrows - row0;
    const int nr = left < rpw ? int(left) : rpw, tot = nr << lx;
    for (int k = 0; k < 3; ++k)
        for (int e = threadIdx.x; e < tot; e += blockDim.x) {
            const int r = e >> lx, i = e & (nx - 1);
            buf[(k * nr + r) * sp + lpos(bitrev(i, lx))] = T[k * ts + (row0 << lx) + e];
        }
    __syncthreads();
    lds_fft(buf, nx, lx, 3 * nr, sp, tws);
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> lx, i = e & (nx - 1);
        const C R = scale * buf[r * sp + lpos(i)], L = scale * buf[(nr + r) * sp + lpos(i)];
        const C Z = scale * buf[(2 * nr + r) * sp + lpos(i)];
        float* f = F + (row0 << lx) + e;
        f[0 * fpl] = float(S(0.5) * (R.re + L.re));
        f[1 * fpl] = float(S(0.5) * (R.im + L.im));
        f[3 * fpl] = float(S(0.5) * (L.im - R.im));
        f[4 * fpl] = float(S(0.5) * (R.re - L.re));
        f[2 * fpl] = float(Z.re);
        f[5 * fpl] = float(Z.im);
    }
}

// ---------------------------------------------------------------- currents (src/sim_particles.cpp:120-158)
//   k_cur_rows   the (1,2,1)/4 zeta filter of the deposit, j_x + i j_y and j_z of a row, x transforms
//   k_cur_cols   y transforms of a tile of columns (S1: in pairs kx, nx - kx), the packed pair unpacked, the filter
// 129 half-cells of 256 x 256: 445 us as filter, two 2D transforms and unpack, now 340 (two transforms move 270 MB each way)
struct CurView {
    int nx, ny, lx, ly, ns, N, a, zf, zu, keep0;
    long nk;
    const double *J, *hc, *filt, *filty;
    const cx *twx, *twy;
    cx *s1, *jx, *jy, *jz;
};
__global__ void __launch_bounds__(kT) k_cur_rows(CurView g, int rpw) {
    extern __shared__ __align__(16) unsigned char smraw[];
    cx* buf = reinterpret_cast<cx*>(smraw);
    const int nx = g.nx, sp = padded(nx);
    cx* tws = buf + size_t(2 * rpw) * sp;
    load_twiddles(tws, g.twx, nx >> 1, false);
    const long row0 = long(blockIdx.x) * rpw, left = (long(g.ns + 1) << g.ly) - row0;
    const int nr = left < rpw ? int(left) : rpw, tot = nr << g.lx, nh = g.ns + 3;
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> g.lx, i = e & (nx - 1);
        const long row = row0 + r;
        const int hk = int(row >> g.ly), hc_ = g.a - 1 + hk, hw = hk + 1;
        const long ip = ((row & (g.ny - 1)) << g.lx) + i;
        double v[3] = {0, 0, 0};
        if (hc_ >= 0 && hc_ <= g.N - 2)
#pragma unroll
            for (int comp = 0; comp < 3; ++comp) {
                const double* Jc = g.J + size_t(comp) * nh * g.nk;
                const double mid = Jc[hw * g.nk + ip];
                if (!g.zf) { v[comp] = mid; continue; }
                const double lo = Jc[(hw - 1) * g.nk + ip], hi = Jc[(hw + 1) * g.nk + ip];
                v[comp] = g.zu ? 0.25 * lo + 0.5 * mid + 0.25 * hi
                               : (0.25 * g.hc[hc_ + 1] * lo + 0.5 * g.hc[hc_ + 2] * mid + 0.25 * g.hc[hc_ + 3] * hi) / g.hc[hc_ + 2];
            }
        const int b = lpos(bitrev(i, g.lx));
        buf[2 * r * sp + b] = mk(v[0], v[1]);
        buf[(2 * r + 1) * sp + b] = mk(v[2], 0);
    }
    __syncthreads();
    lds_fft(buf, nx, g.lx, 2 * nr, sp, tws);
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int r = e >> g.lx, i = e & (nx - 1);
        const long o = (row0 << g.lx) + e;
        g.s1[o] = buf[2 * r * sp + lpos(i)];
        g.jz[o] = buf[(2 * r + 1) * sp + lpos(i)];
    }
}
// The first npair workgroups: 2^lpw column pairs of S1 (pair m: columns m and nx - m, each the other's mirror; m = 0:
// columns 0 and nx/2, each its own); the others: 2 * 2^lpw adjacent columns of j_z
__global__ void __launch_bounds__(kT) k_cur_cols(CurView g, int lpw, long npair) {
    extern __shared__ __align__(16) unsigned char smraw[];
    cx* buf = reinterpret_cast<cx*>(smraw);
    const int ny = g.ny, sp = padded(ny), pw = 1 << lpw;
    cx* tws = buf + size_t(2 * pw) * sp;
    load_twiddles(tws, g.twy, ny >> 1, false);
    const int per = (g.nx / 2) >> lpw;
    const bool pairs = blockIdx.x < npair;
    // the tiles of one XCD consecutive (workgroup b runs on XCD b mod 8): the 64-byte runs of neighbours meet in its L2
    const long w = row_block(int(pairs ? blockIdx.x : blockIdx.x - npair), int(npair), 1), p = w / per;
    const int m0 = int(w - p * per) << lpw, tot = 2 * pw * ny;
    const long pl = p * g.nk;
    auto col = [&](int q) {
        if (!pairs) return 2 * m0 + q;
        const int m = m0 + (q & (pw - 1));
        return q < pw ? m : (m ? g.nx - m : g.nx / 2);
    };
    auto factor = [&](int x, int j) { return (x == 0 && j == 0 && !g.keep0) ? 0.0 : g.filt[x] * g.filty[j]; };
    const cx* A = pairs ? g.s1 : g.jz;
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int j = e >> (lpw + 1), q = e & (2 * pw - 1);
        buf[q * sp + lpos(bitrev(j, g.ly))] = A[pl + (long(j) << g.lx) + col(q)];
    }
    __syncthreads();
    lds_fft(buf, ny, g.ly, 2 * pw, sp, tws);
    for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        const int j = e >> (lpw + 1), q = e & (2 * pw - 1), x = col(q);
        const double f = factor(x, j);
        const long o = pl + (long(j) << g.lx) + x;
        const cx z = buf[q * sp + lpos(j)];
        if (!pairs) { g.jz[o] = f * z; continue; }
        const int qm = m0 + (q & (pw - 1)) ? q ^ pw : q;
        cx X, Y;
        unpack_pair(z, conjg(buf[qm * sp + lpos((ny - j) & (ny - 1))]), X, Y);
        g.jx[o] = f * X; g.jy[o] = f * Y;
    }
}

int ilog(long n) { int l = 0; while ((1L << l) < n) ++l; return l; }
// sequences of length n per workgroup: about kTile values, fewer where the grid would fall below 512 workgroups, at
// least `least` (contiguous runs of a column tile)
int sequences(int n, long total, int least) {
    int q = kTile / n;
    if (q < 1) q = 1;
    while (q > least && total / q < 512) q >>= 1;
    if (q > total) q = int(total);
    return q < 1 ? 1 : q;
}
int lanes(long values) { int t = 64; while (t < values / 8 && t < kT) t <<= 1; return t; }
}  // namespace

void sponge_R(const SpecGeom& g, const FftPlan& p, cx* Rx, cx* Ry, const cx* jkz, const double* hcg, const double* wlo,
              const double* whi, double g2, double opb, const double* mx, const double* mn, const double* mh, cx* S1,
              cx* S2) {
    if (g.ns <= 0) return;
    SpongeView c{};
    c.swap = g.cm;
    c.n0 = g.cm ? g.ny : g.nx; c.n1 = g.cm ? g.nx : g.ny;
    c.l0 = ilog(c.n0); c.l1 = ilog(c.n1);
    c.ns = g.ns; c.N = g.N; c.a = g.a; c.nk = g.nk;
    c.k0 = g.cm ? g.ky : g.kx; c.k1 = g.cm ? g.kx : g.ky;
    c.hc = hcg; c.wl = wlo; c.wu = whi; c.g2 = g2; c.opb = opb; c.jz = jkz;
    c.tw0 = g.cm ? p.twy : p.twx; c.tw1 = g.cm ? p.twx : p.twy;
    c.rx = Rx; c.ry = Ry; c.s1 = S1; c.s2 = S2;
    const long rows = long(c.ns) * c.n1;
    const int rpw = sequences(c.n0, rows, 1);
    hipLaunchKernelGGL(k_sp_rows, dim3(blocks_for(rows, rpw)), dim3(lanes(long(rpw) * c.n0)),
                       (size_t(rpw) * (c.n0 + c.n0 / 8) + c.n0 / 2) * sizeof(cx), stream(), c, rpw);
    const int nc = std::min(sequences(c.n1, long(c.ns) * c.n0, 4), c.n0);
    hipLaunchKernelGGL(k_sp_cols, dim3(unsigned(long(c.ns) * (c.n0 / nc))), dim3(lanes(long(nc) * c.n1)),
                       (size_t(nc) * (c.n1 + c.n1 / 8) + c.n1) * sizeof(cx), stream(), c, ilog(nc), mx, mn, mh,
                       1.0 / (double(g.nx) * g.ny));
    const long pairs = rows / 2;
    int pw = std::max(1, sequences(c.n0, rows, 2) / 2);
    while (pw > 1 && pairs % pw) pw >>= 1;
    hipLaunchKernelGGL(k_sp_unpack, dim3(unsigned(pairs / pw)), dim3(lanes(2L * pw * c.n0)),
                       (size_t(2 * pw) * (c.n0 + c.n0 / 8) + c.n0 / 2) * sizeof(cx), stream(), c, ilog(pw));
    launch_check("sponge");
}

template <class C, class S>
static void real_fields_t(const SpecGeom& g, const FftPlan& p, const cx* Rx, const cx* Ry, const cx* Lx, const cx* Ly,
                          const cx* Ez, const cx* Bz, C* T, long ts, float* F, long fpl, int count) {
    if (count <= 0) return;
    PackView c{{Rx, Lx, Ez}, {Ry, Ly, Bz}, g.nx, g.ny, ilog(g.nx), ilog(g.ny), g.cm, g.nk};
    const int nc = std::min(sequences(g.ny, 3L * count * g.nx, 4), g.nx);
    const long per = long(count) * (g.nx / nc);
    hipLaunchKernelGGL((k_pack_cols<C>), dim3(unsigned(3 * per)), dim3(lanes(long(nc) * g.ny)),
                       (size_t(nc) * (g.ny + g.ny / 8) + g.ny / 2) * sizeof(C), stream(), c, T, ts, ilog(nc), per, p.twy);
    const long rows = long(count) * g.ny;
    const int rpw = std::max(1, sequences(g.nx, 3 * rows, 1) / 3);
    hipLaunchKernelGGL((k_rows_F<C, S>), dim3(blocks_for(rows, rpw)), dim3(lanes(3L * rpw * g.nx)),
                       (size_t(3 * rpw) * (g.nx + g.nx / 8) + g.nx / 2) * sizeof(C), stream(), T, ts, F, fpl, g.nx, c.lx,
                       rows, rpw, p.twx, S(1.0 / (double(g.nx) * g.ny)));
    launch_check("real fields");
}
void real_fields(const SpecGeom& g, const FftPlan& p, const cx* Rx, const cx* Ry, const cx* Lx, const cx* Ly,
                 const cx* Ez, const cx* Bz, cx* T, long ts, float* F, long fpl, int count) {
    real_fields_t<cx, double>(g, p, Rx, Ry, Lx, Ly, Ez, Bz, T, ts, F, fpl, count);
}
void real_fields_f(const SpecGeom& g, const FftPlan& p, const cx* Rx, const cx* Ry, const cx* Lx, const cx* Ly,
                   const cx* Ez, const cx* Bz, cxf* T, long ts, float* F, long fpl, int count) {
    real_fields_t<cxf, float>(g, p, Rx, Ry, Lx, Ly, Ez, Bz, T, ts, F, fpl, count);
}

void current_spectra(const SpecGeom& g, const FftPlan& p, const double* jw, const double* hcg, int zf, int zu, cx* S1,
                     cx* jkx, cx* jky, cx* jkz, int keep0) {
    CurView c{g.nx, g.ny, ilog(g.nx), ilog(g.ny), g.ns, g.N, g.a, zf, zu, keep0, g.nk, jw, hcg, g.filt, g.filty, p.twx, p.twy,
              S1, jkx, jky, jkz};
    const long rows = long(g.ns + 1) * g.ny;
    const int rpw = std::max(1, sequences(g.nx, 2 * rows, 1) / 2);
    hipLaunchKernelGGL(k_cur_rows, dim3(blocks_for(rows, rpw)), dim3(lanes(2L * rpw * g.nx)),
                       (size_t(2 * rpw) * (g.nx + g.nx / 8) + g.nx / 2) * sizeof(cx), stream(), c, rpw);
    int pw = 1;
    while (2 * pw < g.nx / 2 + 1 && 4 * pw * g.ny <= kTile && pw < 8) pw <<= 1;
    const long npair = long(g.ns + 1) * ((g.nx / 2) / pw);
    hipLaunchKernelGGL(k_cur_cols, dim3(unsigned(2 * npair)), dim3(lanes(2L * pw * g.ny)),
                       (size_t(2 * pw) * (g.ny + g.ny / 8) + g.ny / 2) * sizeof(cx), stream(), c, ilog(pw), npair);
    launch_check("current spectra");
}

}  // namespace g3d
