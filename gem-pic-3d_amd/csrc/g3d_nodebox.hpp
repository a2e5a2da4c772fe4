// A workgroup's box of grid nodes, formed from its own particles: lists keep neighbours in space together, so the
// contributions of a workgroup's consecutive particles can be summed in LDS and go to the planes once.
#pragma once
#include "g3d_common.hpp"

namespace g3d {
struct NodeBox {
    int x0, y0, W, H;                // the first node (wrapped); W = 0: no box
};
constexpr int kNodeBoxLanes = 512;   // largest workgroup

// the box of the stencils whose middle nodes are (ix, jn) (of the lanes with on), relative to that of the middle one of the
// first `lanes` lanes so that it may cross the periodic edge (it may be wider than the grid: the first and the last nodes are then the same);
// none beyond cap nodes.  Every lane of the workgroup calls it.
__device__ __forceinline__ NodeBox node_box(bool on, int ix, int jn, int nx, int ny, int lanes, int cap) {
    __shared__ int red[kNodeBoxLanes / 64][4], ref[2];
    if (int(threadIdx.x) == lanes >> 1) { ref[0] = ix; ref[1] = jn; }
    __syncthreads();
    auto near = [](int d, int n) { d = wrap_index(d, n); return d >= n - n / 2 ? d - n : d; };
    int v[4] = {1 << 30, 1 << 30, 1 << 30, 1 << 30};        // minima of u, v, -u, -v
    if (on) { v[0] = near(ix - ref[0], nx); v[1] = near(jn - ref[1], ny); v[2] = -v[0]; v[3] = -v[1]; }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int k = 0; k < 4; ++k) { const int t = __shfl_xor(v[k], o, 64); v[k] = t < v[k] ? t : v[k]; }
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 4; ++k) red[threadIdx.x >> 6][k] = v[k];
    __syncthreads();
    for (int k = 0; k < 4; ++k)
        for (unsigned w = 0; w < blockDim.x / 64; ++w) v[k] = red[w][k] < v[k] ? red[w][k] : v[k];
    if (v[0] == 1 << 30) return NodeBox{0, 0, 0, 0};         // nothing to add
    const int W = -v[2] - v[0] + 3, H = -v[3] - v[1] + 3;
    if (long(W) * H > cap) return NodeBox{0, 0, 0, 0};
    return NodeBox{wrap_index(ref[0] + v[0] - 1, nx), wrap_index(ref[1] + v[1] - 1, ny), W, H};
}
// the middle node of a wrapped coordinate's stencil
__device__ __forceinline__ int mid_node(double x, double d, int n) { return wrap_index(int(floor(x / d + 0.5)), n); }
// node r of the box (row-major): its index in a plane.  The quotient by the reciprocal, (r + 1/2) / W in float, is exact
// for the boxes' at most 2^16 nodes; x0 + u and y0 + v stay below 2 n + 2
__device__ __forceinline__ int box_node(const NodeBox& b, float iw, int r, int nx, int ny) {
    const int v = int((float(r) + 0.5f) * iw);
    int gx = b.x0 + r - v * b.W, gy = b.y0 + v;
    gx -= gx >= nx ? nx : 0; gx -= gx >= nx ? nx : 0;
    gy -= gy >= ny ? ny : 0; gy -= gy >= ny ? ny : 0;
    return gy * nx + gx;
}
}  // namespace g3d
