// What the kernel files share: complex arithmetic, the mode numbering and the
// XCD block order.
#pragma once

#include <hip/hip_runtime.h>

#include "cfg_kernels.hpp"
#include "cfg_lds.hpp"

namespace cfg {

constexpr double PI = 3.14159265358979323846;

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 imul(double s, double2 a) { return make_double2(-(s * a.y), s * a.x); }  // (i s) a

__device__ __forceinline__ int kx_of(const Geom& g, int ikx) { return ikx <= g.kxd ? ikx : ikx - g.nkx; }

constexpr int NXCD = 8;

// The launch's block (x, y, z) renumbered so that each XCD runs a contiguous
// range of the linear block order (x fastest): the dispatcher deals
// consecutive workgroups to the NXCD XCDs in turn, so without it neighbouring
// blocks, which share the cache lines at their edges, fetch those lines into
// different L2s. A permutation of the blocks: the work of each is unchanged.
struct BlockId {
    int x, y, z;
};
__device__ __forceinline__ BlockId xcd_grid() {
    const unsigned gx = gridDim.x, gy = gridDim.y;
    const unsigned T = gx * gy * gridDim.z;
    const unsigned L = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const unsigned q = T / NXCD, r = T % NXCD, x = L % NXCD;
    const unsigned p = x * q + (x < r ? x : r) + L / NXCD;
    const unsigned t = p / gx;
    return BlockId{(int)(p - t * gx), (int)(t % gy), (int)(t / gy)};
}

}  // namespace cfg
