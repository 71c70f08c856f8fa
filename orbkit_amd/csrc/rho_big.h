// Pieces of the many-MO density shared by the contraction of whole 32-row chunks
// (rho_big.hip) and the split-bf16 one, which leaves out a chunk's dead quads of
// rows (rho_big_split.hip).
#pragma once
#include "okmi_internal.h"
#include "split_mfma.h"

namespace {

inline size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

// AO sets of a request (1, 4, 7 or 10)
inline int big_sets(const int* drv_out, int nout)
{
    int mx = 0;
    for (int r = 0; r < nout; ++r) mx = std::max(mx, drv_out[r]);
    return mx == 0 ? 1 : mx <= 3 ? 4 : mx <= 6 ? 7 : 10;
}

// XCD-aware block order: hardware places block b on XCD b % 8; blocks that
// share a point tile (its MO tiles) are given consecutive logical indices on
// one XCD so its L2 serves the AO tile to all of them.
__device__ __forceinline__ int64_t logical_block(int64_t b, int64_t nb)
{
    const int64_t xcd = b & 7, j = b >> 3, per = nb >> 3, rem = nb & 7;
    return (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + j;
}

static __global__ void k_pad_occ_big(const double* occ, int nmo, int mpad, double* out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < mpad) out[i] = i < nmo ? occ[i] : 0.0;
}

struct OutCodes {
    int n;
    int c[16];
};

struct BrickMap {
    int on;
    int64_t bk0, nbx, nby, nbz, nx, ny, nz;
};

// rho[p] = sum_mt partial[mt][0][col]; delta[r][p] = sum_mt partial[mt][c_r][col]
// (code 0: 2 rho, orbkit/core.py:299-300 with drv None).  Column col is point
// p = col (range order) or, in brick order, the grid point of lane col % 64
// of brick bk0 + col / 64 (columns outside the grid are dropped).
static __global__ void k_reduce_big(const double* partial, int nmt, int S, int64_t ld, int64_t np, OutCodes oc,
                             double* rho, double* delta, int64_t ld_delta, BrickMap bm)
{
    const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= np) return;
    int64_t p = col;
    if (bm.on) {
        const int lane = (int)(col & 63);
        int64_t t = bm.bk0 + (col >> 6);
        const int64_t bz = t % bm.nbz;
        t /= bm.nbz;
        const int64_t by = t % bm.nby, bx = t / bm.nby;
        const int64_t ix = 4 * bx + (lane >> 4), iy = 4 * by + ((lane >> 2) & 3), iz = 4 * bz + (lane & 3);
        if (ix >= bm.nx || iy >= bm.ny || iz >= bm.nz) return;
        p = (ix * bm.ny + iy) * bm.nz + iz;
    }
    double r = 0.0;
    for (int m = 0; m < nmt; ++m) r += partial[(int64_t)m * S * ld + col];
    rho[p] = r;
    for (int j = 0; j < oc.n; ++j) {
        const int c = oc.c[j];
        double v = 0.0;
        if (c == 0) {
            v = 2.0 * r;
        } else {
            for (int m = 0; m < nmt; ++m) v += partial[((int64_t)m * S + c) * ld + col];
        }
        delta[j * ld_delta + p] = v;
    }
}

__device__ __forceinline__ double wave_reduce(double v, bool take_min)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double u = __shfl_xor(v, o);
        v = take_min ? fmin(v, u) : fmax(v, u);
    }
    return v;
}

// Bounding box of n columns from col0 on (brick order: the grid points of the
// bricks' lanes; range order: points p0 + column), over a whole wave; columns
// at or past `ncol` and lanes outside the grid are left out (none left: lo > hi).
__device__ __forceinline__ void columns_box(const GridDesc& g, const BrickMap& bm, int64_t p0, int64_t ncol,
                                            int64_t col0, int n, int lane, double (&lo)[3], double (&hi)[3])
{
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        lo[d] = 1e300;
        hi[d] = -1e300;
    }
    for (int j = lane; j < n; j += 64) {
        const int64_t col = col0 + j;
        if (col >= ncol) continue;
        double q[3];
        if (bm.on) {
            const int l = (int)(col & 63);
            int64_t b = bm.bk0 + (col >> 6);
            const int64_t bz = b % bm.nbz;
            b /= bm.nbz;
            const int64_t by = b % bm.nby, bx = b / bm.nby;
            const int64_t ix = 4 * bx + (l >> 4), iy = 4 * by + ((l >> 2) & 3), iz = 4 * bz + (l & 3);
            if (ix >= bm.nx || iy >= bm.ny || iz >= bm.nz) continue;
            q[0] = g.x[ix]; q[1] = g.y[iy]; q[2] = g.z[iz];
        } else {
            grid_point(g, p0 + col, q[0], q[1], q[2]);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = fmin(lo[d], q[d]);
            hi[d] = fmax(hi[d], q[d]);
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        lo[d] = wave_reduce(lo[d], true);
        hi[d] = wave_reduce(hi[d], false);
    }
}

}  // namespace

// the split-bf16 contraction for 1 and 4 AO sets (arguments checked by
// okmi_launch_rho_big)
int okmi_launch_rho_big_split(OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, const double* d_c,
                              const double* d_occ, int nmo, int prec, int S, const int* drv_out, int nout, double* rho,
                              double* delta, int64_t ld_delta, void* ws, size_t ws_bytes, hipStream_t st);
