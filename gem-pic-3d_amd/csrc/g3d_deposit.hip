// Beam deposit in the reference's summation order (src/sim_particles.cpp:56-107).
//
// The reference adds every particle's TSC contributions into jw one particle after the other; with FP64 addition
// the order fixes the last bits, and the start field amplifies them (the relaxation's long step D = 100 dz and the
// near-singular co-moving modes turn 1e-16 into ~1e-12).  Global atomics would sum in schedule order.  Here the
// deposit is a sort instead:
//   1. one lane per particle writes its contribution records: record r = ip R + slot (R = 9 on the Fourier y grid,
//      18 on the free-hand grid: 9 node cells with j_x, j_z and 9 half-node cells with j_y), the cell key
//      (group, half-cell, point) and the values; cells a particle does not touch get the key ~0;
//   2. a stable radix sort of (key, r) groups each cell's records in particle order;
//   3. the values are copied into that order (one lane per record), so that
//   4. one lane per cell (the head of its run of keys) finds the end of its run by bisection; a short run it sums
//      itself from contiguous memory in that order, from zero, as the reference does, and stores the sums into jw;
//   5. a long run (a cell at the core of a dense bunch collects thousands of records) goes to a list, and one wave
//      per long run sums it: the wave loads 64 records at a time with coalesced loads into LDS (the next chunk's
//      loads in flight meanwhile) and one lane adds them in record order (the additions are the same sequence; a
//      lane alone on a long run waited for its loads every few records).
// The result is the reference's single-thread jw, bit for bit.
//
// On a periodic grid of whole 8 x 8 tiles (k_dep_tile) the sort is of particles instead of their 9 records: a particle
// is listed in every (half-cell, tile) bin that its stencil touches (at most 4, 1.6 on average), and a workgroup per bin
// (a wave, for a bin of few) adds the records of its 64 cells in particle order.  2^20 electrons in 128 slices of
// 256 x 256: 1.45 -> 0.48 ms (bins 55 us, sort 130, tiles 282); 2^18 in 256 of 64 x 64: 0.44 -> 0.22 ms.
#include <algorithm>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

#include "g3d_kernels.hpp"
#include "g3d_runtime.hpp"

namespace g3d {
namespace {
constexpr int kT = 256;
// Long lists by radix passes: the default merges up to 2^20 records, a score of launches.  g3d_bunch_currents with keys of 15
// bits, radix and merged: 4000 keys 133 and 94 us, 16384 152 and 113, 65536 157 and 128, 2^18 170 and 195
using DepSort = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config, rocprim::default_config, 0>;
constexpr long kMergeSort = 1L << 17;                // keys up to which the default is used
constexpr unsigned long long kNone = ~0ull;
// key of a record: cell = hw nk + point in the low cb bits (cb: the bits of nh nk), the half-node group in bit cb;
// the sort looks at bits 0 .. cb+1 only, where the empty key ~0 has all ones and so follows every cell

__global__ void __launch_bounds__(kT) k_dep_emit(DepositArgs c, Parts P, long np, int R, int cb,
                                                 unsigned long long* key, unsigned* rec, double* val) {
    const long ip = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (ip >= np) return;
    const long r0 = ip * R;
    for (int s = 0; s < R; ++s) { key[r0 + s] = kNone; rec[r0 + s] = unsigned(r0 + s); }
    if (P.alive[ip] != 1) return;
    int m; double fz;
    c.zax.locate(P.zeta[ip], m, fz);
    const int hw = m - (c.a - 2);
    if (hw < 0 || hw >= c.nh || m < 0 || m > c.N - 2) return;
    const double px = P.px[ip], py = P.py[ip], pz = P.pz[ip];
    const double g = sqrt(1 + px * px + py * py + pz * pz);
    const double vx = px / g, vy = py / g, vz = pz / g;
    const double f = P.q[ip] * P.w[ip] / (c.hcg[m + 2] * c.dx);
    int ix[3], jn[3], jh[3]; double wx[3], wn[3], wh[3];
    tsc_periodic(P.x[ip], c.dx, c.nx, ix, wx);
    const unsigned long long base = (unsigned long long)hw * (unsigned long long)c.nk;
    double* V = val + 3 * r0;
    if (c.yf) {
        tsc_periodic(P.y[ip], c.dy, c.ny, jn, wn);
        for (int v = 0; v < 3; ++v)
            for (int u = 0; u < 3; ++u) {
                const int s = 3 * v + u;
                const double w = f * wx[u] * wn[v] * c.ia[0];
                key[r0 + s] = base + (unsigned long long)(long(jn[v]) * c.nx + ix[u]);
                V[3 * s] = w * vx / vz; V[3 * s + 1] = w * vy / vz; V[3 * s + 2] = w;
            }
        return;
    }
    tsc_freehand(c.yax, P.y[ip], jn, wn, jh, wh);
    for (int v = 0; v < 3; ++v) {
        const bool nod = jn[v] >= 1 && jn[v] <= c.ny - 1, hal = jh[v] >= 0 && jh[v] <= c.ny - 1;
        for (int u = 0; u < 3; ++u) {
            const int s = 3 * v + u;
            if (nod) {
                const double w = f * wx[u] * wn[v] * c.ia[jn[v]];
                key[r0 + s] = base + (unsigned long long)(long(jn[v]) * c.nx + ix[u]);
                V[3 * s] = w * vx / vz; V[3 * s + 1] = 0; V[3 * s + 2] = w;
            }
            if (hal) {
                key[r0 + 9 + s] = (1ull << cb) | (base + (unsigned long long)(long(jh[v]) * c.nx + ix[u]));
                V[3 * (9 + s)] = 0; V[3 * (9 + s) + 2] = 0;
                V[3 * (9 + s) + 1] = f * wx[u] * wh[v] * c.id[jh[v]] * vy / vz;
            }
        }
    }
}

// the values of the sorted records in sorted order
__global__ void __launch_bounds__(kT) k_dep_order(const unsigned long long* key, const unsigned* rec, const double* val,
                                                  long n, double* vs) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n || key[t] == kNone) return;
    const double* v = val + 3 * long(rec[t]);
    vs[3 * t] = v[0]; vs[3 * t + 1] = v[1]; vs[3 * t + 2] = v[2];
}

constexpr int kShortRun = 32;                      // longer runs are summed by a wave each (k_dep_sum_long)

// the sums of one cell into jw
__device__ __forceinline__ void dep_store(unsigned long long k, int cb, double s0, double s1, double s2, double* J,
                                          long nh, long nk, int yf) {
    const bool half = (k >> cb) & 1;
    const long cell = long(k & ((1ull << cb) - 1));
    const long hw = cell / nk, p = cell - hw * nk;
    if (half) { J[(1 * nh + hw) * nk + p] = s1; return; }
    J[(0 * nh + hw) * nk + p] = s0;
    if (yf) J[(1 * nh + hw) * nk + p] = s1;
    J[(2 * nh + hw) * nk + p] = s2;
}

// one lane per sorted record; the head of each run of equal keys sums a short run in record (= particle) order and
// lists a long one
__global__ void __launch_bounds__(kT) k_dep_sum(const unsigned long long* key, const double* vs, long n, double* J,
                                                long nh, long nk, int yf, int cb, long* runs, int* nruns, int cap) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned long long k = key[i];
    if (k == kNone || (i > 0 && key[i - 1] == k)) return;
    long lo = i + 1, hi = n;                        // the run ends at the first record with another key
    while (lo < hi) {
        const long mid = lo + ((hi - lo) >> 1);
        if (key[mid] == k) lo = mid + 1; else hi = mid;
    }
    if (lo - i > kShortRun) {
        const int r = atomicAdd(nruns, 1);
        if (r < cap) { runs[2 * r] = i; runs[2 * r + 1] = lo; return; }
    }
    // in blocks of kU records, the next block's loads in flight during this block's additions (the additions
    // themselves stay in record order)
    constexpr int kU = 8;
    double s0 = 0, s1 = 0, s2 = 0;
    long t = i;
    double a[3 * kU], b[3 * kU];
    if (t + kU <= lo)
        for (int u = 0; u < 3 * kU; ++u) a[u] = vs[3 * t + u];
    while (t + kU <= lo) {
        const long tn = t + kU;
        const bool more = tn + kU <= lo;
        if (more)
            for (int u = 0; u < 3 * kU; ++u) b[u] = vs[3 * tn + u];
        for (int u = 0; u < kU; ++u) { s0 += a[3 * u]; s1 += a[3 * u + 1]; s2 += a[3 * u + 2]; }
        t = tn;
        if (more)
            for (int u = 0; u < 3 * kU; ++u) a[u] = b[u];
    }
    for (; t < lo; ++t) { s0 += vs[3 * t]; s1 += vs[3 * t + 1]; s2 += vs[3 * t + 2]; }
    dep_store(k, cb, s0, s1, s2, J, nh, nk, yf);
}

// one wave per listed long run (persistent: wave w takes runs w, w + waves, ...; every wave leaves when the list is
// done): chunks of 64 records through LDS, lane 0 adds them in record order from zero
constexpr int kRunWaves = 4;                        // waves per workgroup
__global__ void __launch_bounds__(64 * kRunWaves) k_dep_sum_long(const unsigned long long* key, const double* vs,
                                                                 const long* runs, const int* nruns, int cap,
                                                                 double* J, long nh, long nk, int yf, int cb) {
    __shared__ double buf[kRunWaves][2][3 * 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const long waves = long(gridDim.x) * kRunWaves;
    const int nr = min(*nruns, cap);
    for (long r = long(blockIdx.x) * kRunWaves + wv; r < nr; r += waves) {
        const long i = runs[2 * r], lo = runs[2 * r + 1];
        double s0 = 0, s1 = 0, s2 = 0;
        int cur = 0;
        // the first chunk into LDS
        for (int c = lane; c < 3 * 64; c += 64) {
            const long t = i + c / 3;
            buf[wv][0][c] = t < lo ? vs[3 * i + c] : 0.0;
        }
        __builtin_amdgcn_wave_barrier();
        for (long c0 = i; c0 < lo; c0 += 64) {
            // the next chunk's loads in flight while lane 0 adds this one
            double nx[3];
            const long n0 = c0 + 64;
            for (int q = 0; q < 3; ++q) {
                const int c = lane + 64 * q;
                nx[q] = n0 + c / 3 < lo ? vs[3 * n0 + c] : 0.0;
            }
            if (lane == 0) {
                const int m = int(min(long(64), lo - c0));
                const double* b = buf[wv][cur];
                int u = 0;
                // 16 records at a time: their 48 values into registers with one LDS round trip, then the additions
                for (; u + 16 <= m; u += 16) {
                    double w[48];
#pragma unroll
                    for (int q = 0; q < 48; ++q) w[q] = b[3 * u + q];
#pragma unroll
                    for (int q = 0; q < 16; ++q) { s0 += w[3 * q]; s1 += w[3 * q + 1]; s2 += w[3 * q + 2]; }
                }
                for (; u < m; ++u) { s0 += b[3 * u]; s1 += b[3 * u + 1]; s2 += b[3 * u + 2]; }
            }
            for (int q = 0; q < 3; ++q) buf[wv][cur ^ 1][lane + 64 * q] = nx[q];
            cur ^= 1;
            __builtin_amdgcn_wave_barrier();
        }
        if (lane == 0) dep_store(key[i], cb, s0, s1, s2, J, nh, nk, yf);
    }
}

// ---------------------------------------------------------------- particles binned by (half-cell, tile)
constexpr int kDT = 8;                               // cells of a tile each way: one lane per cell
constexpr int kDepSlots = 4;                         // tiles that a 3 x 3 stencil can touch
constexpr int kDepLanes = 512;                       // particles of a chunk
constexpr int kDepWaves = kDepLanes / 64;
constexpr int kDepLong = 512;                        // bins of more particles are taken first
constexpr int kDepFew = 32;                          // bins of at most that many: a wave each (dep_few)
constexpr int kDepPack = 8;                          // doubles per packed particle: xi, yi, f, v_x, v_y, v_z, -, -

// the bins of every particle (slot order = particle order; unused slots: nbin) and what the tiles need of it in one
// 64-byte record (a bin's particles lie anywhere in the list); the counts of k_dep_runs are cleared on the way
__global__ void __launch_bounds__(kT) k_dep_bins(DepositArgs c, Parts P, long np, int ntx, int nty, unsigned nbin,
                                                 unsigned* key, double* pack, int* cnt) {
    const long ip = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (ip < 3) cnt[ip] = 0;
    if (ip >= np) return;
    unsigned k[kDepSlots] = {nbin, nbin, nbin, nbin};
    int m = 0; double fz;
    int hw = -1;
    if (P.alive[ip] == 1) {
        c.zax.locate(P.zeta[ip], m, fz);
        hw = m - (c.a - 2);
        if (m < 0 || m > c.N - 2 || hw >= c.nh) hw = -1;
    }
    if (hw >= 0) {
        const double px = P.px[ip], py = P.py[ip], pz = P.pz[ip];
        const double g = sqrt(1 + px * px + py * py + pz * pz);
        const double xi = P.x[ip] / c.dx, yi = P.y[ip] / c.dy;
        int ix[3], jn[3]; double w[3];
        tsc_w(xi, ix, w);
        tsc_w(yi, jn, w);
        const int xa = wrap_index(ix[0], c.nx) / kDT, xb = wrap_index(ix[2], c.nx) / kDT;
        const int ya = wrap_index(jn[0], c.ny) / kDT, yb = wrap_index(jn[2], c.ny) / kDT;
        const unsigned base = unsigned(hw) * unsigned(nty * ntx);
        k[0] = base + unsigned(ya * ntx + xa);
        if (xb != xa) k[1] = base + unsigned(ya * ntx + xb);
        if (yb != ya) {
            k[2] = base + unsigned(yb * ntx + xa);
            if (xb != xa) k[3] = base + unsigned(yb * ntx + xb);
        }
        double2* q = reinterpret_cast<double2*>(pack + kDepPack * ip);
        q[0] = make_double2(xi, yi);
        q[1] = make_double2(P.q[ip] * P.w[ip] / (c.hcg[m + 2] * c.dx), px / g);
        q[2] = make_double2(py / g, pz / g);
    }
    *reinterpret_cast<uint4*>(key + kDepSlots * ip) = make_uint4(k[0], k[1], k[2], k[3]);
}
// the runs of equal keys, (first record, end) each: in the first `cap` slots of `bins` the long ones from the front and
// those of more than kDepFew records from the back, from slot cap on the others (cnt: the three numbers)
__global__ void __launch_bounds__(kT) k_dep_runs(const unsigned* key, long n, unsigned nbin, long* bins, int* cnt, int cap) {
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned k = key[i];
    if (k >= nbin || (i > 0 && key[i - 1] == k)) return;
    long lo = i + 1, hi = n;
    // the end by doubling steps, then bisection (most runs are short)
    for (long st = 8; lo < hi; st <<= 1) {
        const long t = i + st;
        if (t >= hi) break;
        if (key[t] == k) lo = t + 1; else { hi = t; break; }
    }
    while (lo < hi) {
        const long mid = lo + ((hi - lo) >> 1);
        if (key[mid] == k) lo = mid + 1; else hi = mid;
    }
    // every run has its slot: runs <= cap.  One address per branch: the compiler then adds once per wave
    long slot;
    if (lo - i > kDepLong) slot = atomicAdd(&cnt[0], 1);
    else if (lo - i > kDepFew) slot = long(cap) - 1 - atomicAdd(&cnt[1], 1);
    else slot = long(cap) + atomicAdd(&cnt[2], 1);
    bins[2 * slot] = i; bins[2 * slot + 1] = lo;
}
// x / d with r = 1 / d: the quotient estimate and one exact correction, as the compiler's division ends, with div_fixup for
// infinities and NaN (the scaling for extreme exponents is left out)
__device__ __forceinline__ double div_by(double x, double d, double r) {
    const double q = x * r;
    return __builtin_amdgcn_div_fixup(fma(fma(-q, d, x), r, q), d, x);
}
constexpr int kFewRec = 11;                          // doubles per particle: f w_x (3), w_y (3), v_x, v_y, v_z, 1/v_z, first nodes
// A bin of at most kDepFew particles by one wave, B: kDepFew records of LDS: the particles' stencils formed by a lane each
// and left there, then one lane per cell of the tile takes the particles in list order.  A workgroup of k_dep_tile fills a CU
// with its lists, so 256 bins went through at a time however few their particles.  Electrons anywhere in 128 slices of 16 x 512
// points, all of g3d_bunch_currents, with a workgroup for every bin, now, and by the record sort (8 x 1024 points): 16384
// electrons 441, 130 and 168 us; 65536 538, 187 and 288; 2^18 565, 304 and 440; 10^5 in 256 x 256 2580 and 610.  In a launch
// of their own the small bins take up to 20 us less there, but bunches pay for it (65536 171 us, here 167); so launched,
// kDepFew 16, 32 and 64: 2^18 anywhere 453, 293 and 268 us, a bunch of 2^18 236, 237 and 241
__device__ __forceinline__ void dep_few(const DepositArgs& c, const unsigned* key, const unsigned* rec, const double* pack,
                                        const long* bins, int cap, int b, int ntx, int nty, double* B) {
    const int lane = threadIdx.x & 63;
    const long lo = bins[2 * (long(cap) + b)];
    const int m = int(bins[2 * (long(cap) + b) + 1] - lo);
    const unsigned k = key[lo];
    const int tile = int(k % unsigned(ntx * nty)), hw = int(k / unsigned(ntx * nty));
    const int x0 = (tile % ntx) * kDT, y0 = (tile / ntx) * kDT;
    if (lane < m) {
        const double2* q = reinterpret_cast<const double2*>(pack + kDepPack * long(rec[lo + lane] / kDepSlots));
        const double2 q0 = q[0], q1 = q[1], q2 = q[2];
        int ix[3], jn[3]; double wx[3], wn[3];
        tsc_w(q0.x, ix, wx);
        tsc_w(q0.y, jn, wn);
        double* r = B + kFewRec * lane;
#pragma unroll
        for (int u = 0; u < 3; ++u) { r[u] = q1.x * wx[u]; r[3 + u] = wn[u]; }
        r[6] = q1.y; r[7] = q2.x; r[8] = q2.y; r[9] = 1 / q2.y;
        reinterpret_cast<int2*>(r + 10)[0] = make_int2(wrap_index(ix[0], c.nx), wrap_index(jn[0], c.ny));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int x = x0 + (lane & (kDT - 1)), y = y0 + lane / kDT;
    double a0 = 0, a1 = 0, a2 = 0;
    // no branch: a particle that misses the cell adds zero, which never changes a sum that began as +0
#pragma unroll 4
    for (int t = 0; t < m; ++t) {
        const double* r = B + kFewRec * t;
        const int2 n0 = reinterpret_cast<const int2*>(r + 10)[0];
        int u = x - n0.x, v = y - n0.y;
        u += u < 0 ? c.nx : 0;
        v += v < 0 ? c.ny : 0;
        const bool in = u < 3 && v < 3;
        const double w = r[in ? u : 0] * r[3 + (in ? v : 0)] * c.ia[0], vz = r[8], rz = r[9];
        const double p0 = div_by(w * r[6], vz, rz), p1 = div_by(w * r[7], vz, rz);
        a0 += in ? p0 : 0.0;
        a1 += in ? p1 : 0.0;
        a2 += in ? w : 0.0;
    }
    double* J = c.J + long(hw) * c.nk + long(y) * c.nx + x;
    const long pl = long(c.nh) * c.nk;
    J[0] = a0; J[pl] = a1; J[2 * pl] = a2;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();                  // before the next bin's records
}
// One workgroup per bin (persistent), then the bins of few.  A chunk of kDepLanes particles at a time, in list order: which of the tile's 8
// columns and 8 rows a particle's stencil covers, as ballots over the wave; the product of a column's and a row's ballot
// is the set of the cell's particles, so its population below a lane is the particle's rank in the cell's list.
// Every record goes to its place in the list of its cell in LDS, and wave k < 3 adds component k, one lane per cell,
// in list order.  The next chunk's particles are loaded during the additions.  The chain is the densest cell's
// additions from LDS.
__global__ void __launch_bounds__(kDepLanes) k_dep_tile(DepositArgs c, const unsigned* key, const unsigned* rec,
                                                        const double* pack, const long* bins, const int* cnt, int cap,
                                                        int ntx, int nty) {
    __shared__ __align__(16) double vals[3][9 * kDepLanes + 64];
    __shared__ unsigned long long bal[kDepWaves][2 * kDT];
    __shared__ int count[kDepWaves][64], start[kDepWaves][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int nl = cnt[0], nb = nl + cnt[1];
    for (int b = blockIdx.x; b < nb; b += gridDim.x) {
        const long slot = b < nl ? b : long(cap) - 1 - (b - nl);
        const long lo = bins[2 * slot], hi = bins[2 * slot + 1];
        const unsigned k = key[lo];
        const int tile = int(k % unsigned(ntx * nty)), hw = int(k / unsigned(ntx * nty));
        const int x0 = (tile % ntx) * kDT, y0 = (tile / ntx) * kDT;
        double acc = 0;
        double2 q0{}, q1{}, q2{};
        unsigned rn = 0;                              // the record of the chunk after the loaded one
        auto load = [&](long t) {
            const double2* q = reinterpret_cast<const double2*>(pack + kDepPack * long(rn / kDepSlots));
            if (t < hi) { q0 = q[0]; q1 = q[1]; q2 = q[2]; }
            if (t + kDepLanes < hi) rn = rec[t + kDepLanes];
        };
        if (lo + threadIdx.x < hi) rn = rec[lo + threadIdx.x];
        load(lo + threadIdx.x);
        for (long t0 = lo; t0 < hi; t0 += kDepLanes) {
            const bool on = t0 + threadIdx.x < hi;
            int ix[3], jn[3]; double wx[3], wn[3];
            tsc_w(q0.x, ix, wx);
            tsc_w(q0.y, jn, wn);
            const double f = q1.x, vx = q1.y, vy = q2.x, vz = q2.y, rz = 1 / vz;
            unsigned cols = 0, rows = 0;
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                ix[u] = wrap_index(ix[u], c.nx) - x0; jn[u] = wrap_index(jn[u], c.ny) - y0;
                if (on && ix[u] >= 0 && ix[u] < kDT) cols |= 1u << ix[u]; else ix[u] = -1;
                if (on && jn[u] >= 0 && jn[u] < kDT) rows |= 1u << jn[u]; else jn[u] = -1;
            }
#pragma unroll
            for (int u = 0; u < kDT; ++u) {
                const unsigned long long mx = __ballot(cols >> u & 1u), my = __ballot(rows >> u & 1u);
                if (lane == u) { bal[wv][u] = mx; bal[wv][kDT + u] = my; }
            }
            __syncthreads();                          // also: the previous chunk's additions are done
            count[wv][lane] = int(__popcll(bal[wv][lane & (kDT - 1)] & bal[wv][kDT + lane / kDT]));
            __syncthreads();
            // every wave for itself: the lists' places (cell order, then wave order within a cell)
            int tot = 0, mine = 0;
#pragma unroll
            for (int w = 0; w < kDepWaves; ++w) {
                if (w == wv) mine = tot;
                tot += count[w][lane];
            }
            const int room = (tot + 1) & ~1;          // every list on an even place: read two records at a time
            int inc = room;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(inc, d, 64);
                if (lane >= d) inc += o;
            }
            const int base = inc - room;
            start[wv][lane] = base + mine;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int v = 0; v < 3; ++v)
#pragma unroll
                for (int u = 0; u < 3; ++u) {
                    if (ix[u] < 0 || jn[v] < 0) continue;
                    const int cell = jn[v] * kDT + ix[u];
                    const unsigned long long mk_ = bal[wv][ix[u]] & bal[wv][kDT + jn[v]];
                    const int pos = start[wv][cell] + __builtin_amdgcn_mbcnt_hi(unsigned(mk_ >> 32),
                                                                                 __builtin_amdgcn_mbcnt_lo(unsigned(mk_), 0));
                    const double w = f * wx[u] * wn[v] * c.ia[0];
                    vals[0][pos] = div_by(w * vx, vz, rz);
                    vals[1][pos] = div_by(w * vy, vz, rz);
                    vals[2][pos] = w;
                }
            load(t0 + kDepLanes + threadIdx.x);
            __syncthreads();
            if (wv < 3) {
                // two groups of 8 records in turn, the next group's reads in flight during this one's additions
                const double* l = vals[wv] + base;
                auto get = [&](double2 (&r)[4], int at) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) r[u] = *reinterpret_cast<const double2*>(l + at + 2 * u);
                };
                auto add = [&](const double2 (&r)[4]) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) { acc += r[u].x; acc += r[u].y; }
                };
                double2 ra[4], rb[4];
                int m = 0;
                if (tot >= 8) get(ra, 0);
                while (m + 24 <= tot) {
                    get(rb, m + 8);
                    add(ra);
                    get(ra, m + 16);
                    add(rb);
                    m += 16;
                }
                if (m + 8 <= tot) {
                    if (m + 16 <= tot) get(rb, m + 8);
                    add(ra);
                    m += 8;
                    if (m + 8 <= tot) { add(rb); m += 8; }
                }
                for (; m < tot; ++m) acc += l[m];
            }
        }
        if (wv < 3)
            c.J[(long(wv) * c.nh + hw) * c.nk + long(y0 + lane / kDT) * c.nx + x0 + (lane & (kDT - 1))] = acc;
        __syncthreads();                              // before the next bin's ballots and lists
    }
    // the bins of few particles too, a wave each, from the last workgroup (which had no other bin) on
    for (int b = (int(gridDim.x) - 1 - int(blockIdx.x)) * kDepWaves + wv; b < cnt[2]; b += int(gridDim.x) * kDepWaves)
        dep_few(c, key, rec, pack, bins, cap, b, ntx, nty, &vals[0][0] + wv * (kDepFew * kFewRec));
}

// Every buffer by its own length: the two sorts share some of them, and each needs other lengths of them
template <class T> void fit(DevBuf<T>& b, long n) {
    if (b.size() < size_t(n)) b.resize(size_t(n) + size_t(n) / 4);
}

// from which sizes the particle sort runs: whole tiles on a periodic grid, keys and records in 32 bits
bool tiled_deposit(const DepositArgs& a, long np, unsigned& nbin) {
    if (!a.yf || a.nx % kDT || a.ny % kDT || a.nx < 2 * kDT || a.ny < 2 * kDT || np > (1L << 28)) return false;
    const long n = long(a.nh) * (a.nx / kDT) * (a.ny / kDT);
    if (n >= (1L << 30)) return false;
    nbin = unsigned(n);
    return true;
}
void tiled_deposit_run(const DepositArgs& a, Parts p, long np, unsigned nbin, DepositScratch& s) {
    const int ntx = a.nx / kDT, nty = a.ny / kDT;
    const long n = np * kDepSlots;
    unsigned bits = 1;
    while ((1ull << bits) <= nbin) ++bits;            // the unused slots' key nbin among them
    fit(s.k0, n); fit(s.k1, n); fit(s.rec1, n);
    fit(s.val, kDepPack * np);
    const int cap = int(std::min<long>(n, long(nbin)));
    fit(s.runs, 4L * cap);
    fit(s.nruns, 3);
    hipLaunchKernelGGL(k_dep_bins, dim3(blocks_for(np, kT)), dim3(kT), 0, stream(), a, p, np, ntx, nty, nbin, s.k0.data(),
                       s.val.data(), s.nruns.data());
    const rocprim::counting_iterator<unsigned> ids(0);
    auto sort = [&](auto config) {
        size_t bytes = 0;
        hip_check(rocprim::radix_sort_pairs<decltype(config)>(nullptr, bytes, s.k0.data(), s.k1.data(), ids, s.rec1.data(), n, 0, bits,
                                                              stream()), "beam deposit sort size");
        if (s.tmp.size() < bytes) s.tmp.resize(bytes + bytes / 4 + 256);
        bytes = s.tmp.size();
        hip_check(rocprim::radix_sort_pairs<decltype(config)>(s.tmp.data(), bytes, s.k0.data(), s.k1.data(), ids, s.rec1.data(), n, 0,
                                                              bits, stream()), "beam deposit sort");
    };
    if (n <= kMergeSort) sort(rocprim::default_config{});
    else sort(DepSort{});
    hipLaunchKernelGGL(k_dep_runs, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), s.k1.data(), n, nbin, s.runs.data(),
                       s.nruns.data(), cap);
    hipLaunchKernelGGL(k_dep_tile, dim3(unsigned(std::min(cap, 1024))), dim3(kDepLanes), 0, stream(), a, s.k1.data(),
                       s.rec1.data(), s.val.data(), s.runs.data(), s.nruns.data(), cap, ntx, nty);
    launch_check("beam deposit (tiles)");
}
}  // namespace

void bunch_deposit(const DepositArgs& a, Parts p, long np, DepositScratch& s) {
    if (np <= 0) return;
    unsigned nbin = 0;
    if (tiled_deposit(a, np, nbin)) { tiled_deposit_run(a, p, np, nbin, s); return; }
    const int R = a.yf ? 9 : 18;
    const long n = np * R;
    if (n > long(0xffffffffu)) throw std::runtime_error("beam deposit: too many contribution records");
    int cb = 1;                                     // the bits of the cells hw nk + point
    while ((1ull << cb) < (unsigned long long)a.nh * (unsigned long long)a.nk) ++cb;
    if (cb > 60) throw std::runtime_error("beam deposit: grid too large");
    fit(s.key0, n); fit(s.key1, n); fit(s.rec0, n); fit(s.rec1, n);
    fit(s.val, 3 * n); fit(s.vs, 3 * n);
    hipLaunchKernelGGL(k_dep_emit, dim3(blocks_for(np, kT)), dim3(kT), 0, stream(), a, p, np, R, cb, s.key0.data(),
                       s.rec0.data(), s.val.data());
    launch_check("beam deposit records");
    // bits 0 .. cb+1: the cell, the group bit, and above every valid key the low bits of the empty key ~0
    const unsigned end_bit = unsigned(cb) + 2;
    size_t bytes = 0;
    hip_check(rocprim::radix_sort_pairs(nullptr, bytes, s.key0.data(), s.key1.data(), s.rec0.data(), s.rec1.data(),
                                        n, 0, end_bit, stream()), "beam deposit sort size");
    if (s.tmp.size() < bytes) s.tmp.resize(bytes + bytes / 4 + 256);
    bytes = s.tmp.size();
    hip_check(rocprim::radix_sort_pairs(s.tmp.data(), bytes, s.key0.data(), s.key1.data(), s.rec0.data(),
                                        s.rec1.data(), n, 0, end_bit, stream()), "beam deposit sort");
    hipLaunchKernelGGL(k_dep_order, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), s.key1.data(), s.rec1.data(),
                       s.val.data(), n, s.vs.data());
    // long runs: at most one per kShortRun + 1 records
    const int cap = int(n / (kShortRun + 1) + 1);
    fit(s.runs, 2L * cap);
    fit(s.nruns, 1);
    hip_check(hipMemsetAsync(s.nruns.data(), 0, sizeof(int), stream()), "hipMemsetAsync");
    hipLaunchKernelGGL(k_dep_sum, dim3(blocks_for(n, kT)), dim3(kT), 0, stream(), s.key1.data(), s.vs.data(), n, a.J,
                       long(a.nh), a.nk, a.yf, cb, s.runs.data(), s.nruns.data(), cap);
    hipLaunchKernelGGL(k_dep_sum_long, dim3(1024), dim3(64 * kRunWaves), 0, stream(), s.key1.data(), s.vs.data(),
                       s.runs.data(), s.nruns.data(), cap, a.J, long(a.nh), a.nk, a.yf, cb);
    launch_check("beam deposit sums");
}

}  // namespace g3d
