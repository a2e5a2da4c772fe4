// March kernels: every mode from the front slice to the rear (one lane per mode, slice n+1 carried in registers,
// the explicit inputs of the next slice prefetched while the current one is computed), and one slice.
#include <cstdlib>
#include "g3d_kernels.hpp"
#include "g3d_march_half.hpp"
#include "g3d_runtime.hpp"

namespace g3d {
namespace {

__device__ __forceinline__ Mode6 load6(const MarchView& c, long o) {
    return Mode6{c.Rx[o], c.Ry[o], c.Ez[o], c.Bz[o], c.Lx[o], c.Ly[o]};
}
__device__ __forceinline__ void store6(const MarchView& c, long o, const Mode6& m) {
    c.Rx[o] = m.Rx; c.Ry[o] = m.Ry; c.Ez[o] = m.Ez; c.Bz[o] = m.Bz; c.Lx[o] = m.Lx; c.Ly[o] = m.Ly;
}

// workgroups of one wave for the march of every mode, so that a small grid (64 x 64 modes: 64 waves) spreads
// over as many compute units
constexpr int kMarchT = 64;
// slices hi-1 ... lo of every mode (src/sim_fields.cpp:7-31, Fourier y), one lane per mode
__global__ void __launch_bounds__(kMarchT) k_march_all(MarchView c, int lo, int hi) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= c.nk) return;
    int ixx, j;
    mode_xy(c, i, ixx, j);
    // the wavenumbers once and the slice weights with the slice's data, ahead of it: a load issued inside the
    // chain would wait, in the in-order memory counter, for the stores of the slice before it
    const double kxv = c.kx[ixx], kyv = c.ky[j];
    Mode6 up{};
    if (hi < c.N) up = load6(c, long(hi - c.a) * c.nk + i);
    // the explicit part and the currents of the next slice are loaded while this slice is marched (the march of
    // a mode is a chain over the slices: each load on it would add its latency to every slice)
    long o = long(hi - 1 - c.a) * c.nk + i;
    Mode6 old{c.Rx[o], c.Ry[o], c.Ez[o], c.Bz[o], {}, {}};
    Cur9 cur = load_cur(c, i, hi - 1);
    SliceW w = slice_w(c, hi - 1);
    for (int n = hi - 1; n >= lo; --n) {
        Mode6 nxt{};
        Cur9 curn{};
        SliceW wn{};
        const long on = o - c.nk;
        if (n > lo) {
            nxt.Rx = c.Rx[on]; nxt.Ry = c.Ry[on]; nxt.Ez = c.Ez[on]; nxt.Bz = c.Bz[on];
            curn = load_cur(c, i, n - 1);
            wn = slice_w(c, n - 1);
        }
        up = march_mode_k(c, kxv, kyv, w, n, old, up, cur);
        store6(c, o, up);
        old = nxt;
        cur = curn;
        w = wn;
        o = on;
    }
}

// The same march with its inputs staged in LDS, for grids of few modes, where the chain of one wave over the slices is
// the whole kernel.  Two lanes per mode, one real half-system each (g3d_march_half.hpp).  Wave 0 of a workgroup
// marches 32 modes slice by slice, reading only LDS and storing the results, while waves 1-3 load the inputs of the
// next block of kStageB slices, form the explicit parts of R from them and write those and the currents into the other
// of two LDS buffers (so the loads are issued a block ahead and never wait behind the marching wave's stores).  What
// is left on the chain is about 90 FP64 operations per slice: 64 x 64 x 256 modes and slices in 106 us, with one
// lane per mode and its complex arithmetic 216 us.
constexpr int kStageB = 6;
constexpr int kStageT = 256;
constexpr int kStageProd = kStageT / 64 - 1;         // producer waves
constexpr int kStagePer = kStageB / kStageProd;      // slices of a block per producer wave
static_assert(kStagePer * kStageProd == kStageB, "march staging: whole slices per producer wave");
constexpr int kStageComp = 5;                        // R_sx, R_sy, jk_x, jk_y, jk_z (the last three of half-cell n)
constexpr size_t kStageLds = size_t(2) * kStageB * (kStageComp * 64 + 1) * sizeof(double);
constexpr long kStageMaxModes = 16384;

// the inputs of one slice for one lane: what the explicit part needs, before the arithmetic
struct StageIn {
    double Rx, Ry, Ez, Bz, j0x[2], j0y[2], jkx[2], jky[2], jkz, wl, wu, h;
};
__device__ __forceinline__ void stage_load(const MarchView& c, int n, long p, long e, StageIn& r) {
    const long o = 2 * long(n - c.a) * c.nk, pl = 2 * c.nk;
    r.Rx = dbl(c.Rx)[o + p]; r.Ry = dbl(c.Ry)[o + p]; r.Ez = dbl(c.Ez)[o + e]; r.Bz = dbl(c.Bz)[o + e];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const long q = o + u * pl + p;
        r.j0x[u] = dbl(c.j0x)[q]; r.j0y[u] = dbl(c.j0y)[q]; r.jkx[u] = dbl(c.jkx)[q]; r.jky[u] = dbl(c.jky)[q];
    }
    r.jkz = dbl(c.jkz)[o + pl + e];
    const SliceW w = slice_w(c, n);
    r.wl = w.wl; r.wu = w.wu; r.h = w.h;
}
__device__ __forceinline__ void stage_write(double* q, double* hs, int lane, const HalfK& k, double D, const StageIn& r) {
    double Rsx, Rsy;
    half_explicit(k, D, r.wl, r.wu, r.Rx, r.Ry, r.Ez, r.Bz, r.j0x, r.j0y, r.jkx, r.jky, Rsx, Rsy);
    q[lane] = Rsx; q[64 + lane] = Rsy; q[128 + lane] = r.jkx[1]; q[192 + lane] = r.jky[1]; q[256 + lane] = r.jkz;
    if (lane == 0) *hs = r.h;
}

// slices hi-1 ... lo of every mode, 32 modes per workgroup of kStageT lanes (blocks of kStageB slices: block b
// holds slices hi-1-b kStageB ... down to lo)
__global__ void __launch_bounds__(kStageT) k_march_staged(MarchView c, int lo, int hi) {
    extern __shared__ __align__(16) double stg[];
    double* hst = stg + 2 * kStageB * kStageComp * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane & 1;
    const long i = long(blockIdx.x) * 32 + (lane >> 1);
    const bool on = i < c.nk;
    const long ic = on ? i : c.nk - 1, p = 2 * ic + half, e = 2 * ic + 1 - half;
    int ixx, j;
    mode_xy(c, ic, ixx, j);
    const HalfK k = half_k(half, c.kx[ixx], c.ky[j]);
    const int nblk = (hi - lo + kStageB - 1) / kStageB;
    if (wave > 0) {
        // a producer's block b + 1 is written in the interval of block b from registers loaded in the interval
        // before, so each block's loads have two march intervals to arrive (slices below lo load slice lo, never read)
        const int s0 = (wave - 1) * kStagePer;
        StageIn r[kStagePer];
        auto load = [&](int b) {
#pragma unroll
            for (int q = 0; q < kStagePer; ++q) stage_load(c, max(hi - 1 - b * kStageB - s0 - q, lo), p, e, r[q]);
        };
        auto write = [&](int b) {
#pragma unroll
            for (int q = 0; q < kStagePer; ++q) {
                const int s = (b & 1) * kStageB + s0 + q;
                stage_write(stg + s * kStageComp * 64, hst + s, lane, k, c.D, r[q]);
            }
        };
        load(0);
        write(0);
        if (nblk > 1) load(1);
        for (int b = 0; b < nblk; ++b) {
            __syncthreads();             // buffer b & 1 staged; the other one read by the march of block b - 1
            if (b + 1 < nblk) write(b + 1);
            if (b + 2 < nblk) load(b + 2);
        }
        return;
    }
    Half6 up{};
    if (hi < c.N) {
        const long o = 2 * long(hi - c.a) * c.nk;
        up = Half6{dbl(c.Rx)[o + p], dbl(c.Ry)[o + p], dbl(c.Ez)[o + e], dbl(c.Bz)[o + e], dbl(c.Lx)[o + p], dbl(c.Ly)[o + p]};
    }
    HalfDen dn{};
    for (int b = 0; b < nblk; ++b) {
        __syncthreads();
        for (int s = 0; s < kStageB; ++s) {
            const int n = hi - 1 - b * kStageB - s;
            if (n < lo) break;
            const int sb = (b & 1) * kStageB + s;
            const double* q = stg + sb * kStageComp * 64 + lane;
            const double Rsx = q[0], Rsy = q[64], jx = q[128], jy = q[192], jz = q[256], h = hst[sb];
            if (n == c.N - 1) up = Half6{Rsx, Rsy, 0, 0, 0, 0};      // front of the window: L = E_z = B_z = 0
            else {
                dn.set(k, h, c.D);
                up = half_implicit(k, dn, c.D, h, Rsx, Rsy, jx, jy, jz, up);
            }
            if (on) {
                const long o = 2 * long(n - c.a) * c.nk;
                dbl(c.Rx)[o + p] = up.Rx; dbl(c.Ry)[o + p] = up.Ry; dbl(c.Ez)[o + e] = up.Ez; dbl(c.Bz)[o + e] = up.Bz;
                dbl(c.Lx)[o + p] = up.Lx; dbl(c.Ly)[o + p] = up.Ly;
            }
        }
    }
}

// one slice n; bk* optional: restore = 0 saves slice n before the update, restore = 1 reads it from there
__global__ void __launch_bounds__(256) k_march_slice(MarchView c, int n, cx* bRx, cx* bRy, cx* bEz, cx* bBz,
                                                     int restore) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= c.nk) return;
    const long o = long(n - c.a) * c.nk + i;
    Mode6 old;
    if (restore && bRx) { old.Rx = bRx[i]; old.Ry = bRy[i]; old.Ez = bEz[i]; old.Bz = bBz[i]; }
    else {
        old.Rx = c.Rx[o]; old.Ry = c.Ry[o]; old.Ez = c.Ez[o]; old.Bz = c.Bz[o];
        if (bRx) { bRx[i] = old.Rx; bRy[i] = old.Ry; bEz[i] = old.Ez; bBz[i] = old.Bz; }
    }
    Mode6 up{};
    if (n < c.N - 1) up = load6(c, o + c.nk);
    store6(c, o, march_mode(c, i, n, old, up));
}

MarchView view_of(const g3d_march_ctx& m) {
    MarchView v;
    v.Rx = m.Rx; v.Ry = m.Ry; v.Ez = m.Ez; v.Bz = m.Bz; v.Lx = m.Lx; v.Ly = m.Ly;
    v.j0x = m.j0x; v.j0y = m.j0y; v.jkx = m.jkx; v.jky = m.jky; v.jkz = m.jkz;
    v.kx = m.kx; v.ky = m.ky; v.hcg = m.hcg; v.wlo = m.wlo; v.whi = m.whi;
    v.D = m.D; v.a = m.a; v.N = m.N; v.nx = m.nx; v.nk = m.nk; v.ny = m.ny;
    return v;
}
void require_one_gpu(const g3d_march_ctx& m) {
    if (m.a != 0 || m.b != m.N) throw std::runtime_error("g3d march: one GPU owns all slices (a = 0, b = N)");
    if (!m.ky && (!m.scp || !m.iD || !m.iA || m.ny < 4))
        throw std::runtime_error("g3d march: the free-hand y march needs iD, iA, scp (2 nk doubles) and ny >= 4");
}
LineView lines_of(const g3d_march_ctx& m) {
    LineView L;
    L.mv = view_of(m); L.iD = m.iD; L.iA = m.iA; L.scp = m.scp; L.ny = m.ny; L.piv = nullptr;
    return L;
}
}  // namespace

void march_all(const MarchView& v, int lo, int hi) {
    if (hi <= lo) return;
    // the staged march up to two workgroups per compute unit (128 x 128 modes); G3D_MARCH_STAGED=0 turns it off
    const char* e = getenv("G3D_MARCH_STAGED");
    if ((e ? atoi(e) : 1) && v.nk <= kStageMaxModes)
        hipLaunchKernelGGL(k_march_staged, dim3(blocks_for(v.nk, 32)), dim3(kStageT), kStageLds, stream(), v, lo, hi);
    else
        hipLaunchKernelGGL(k_march_all, dim3(blocks_for(v.nk, kMarchT)), dim3(kMarchT), 0, stream(), v, lo, hi);
    launch_check("march");
}
void march_one(const MarchView& v, int n, cx* bRx, cx* bRy, cx* bEz, cx* bBz, int restore) {
    hipLaunchKernelGGL(k_march_slice, dim3(blocks_for(v.nk, 256)), dim3(256), 0, stream(), v, n, bRx, bRy, bEz, bBz,
                       restore);
    launch_check("march slice");
}

}  // namespace g3d

extern "C" {
int g3d_march(const g3d_march_ctx* c, int lo, int hi) {
    return g3d::guard([&] {
        g3d::require_one_gpu(*c);
        if (c->ky) g3d::march_all(g3d::view_of(*c), lo, hi);
        else g3d::march_lines(g3d::lines_of(*c), lo, hi);
    });
}
int g3d_march_slice(const g3d_march_ctx* c, int n, int restore) {
    return g3d::guard([&] {
        g3d::require_one_gpu(*c);
        if (c->ky) {
            g3d::march_one(g3d::view_of(*c), n, c->bkRx, c->bkRy, c->bkEz, c->bkBz, restore);
            return;
        }
        if (c->bkRx) {                     // the backup of slice n, then the lines of slice n
            const long o = long(n - c->a) * c->nk;
            g3d::cx* sl[4] = {c->Rx + o, c->Ry + o, c->Ez + o, c->Bz + o};
            g3d::cx* bk[4] = {c->bkRx, c->bkRy, c->bkEz, c->bkBz};
            for (int k = 0; k < 4; ++k) {
                if (restore) g3d::copy_planes(sl[k], bk[k], c->nk);
                else g3d::copy_planes(bk[k], sl[k], c->nk);
            }
        }
        g3d::march_lines(g3d::lines_of(*c), n, n + 1);
    });
}
}
