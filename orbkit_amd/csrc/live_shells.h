// Per-tile lists of the shells in reach, for the FP64 kernels that contract
// only those: a 64-point brick reaches about a quarter of the AO rows of a
// 20-atom molecule and 7% of those of 200 atoms, where fixed 32-row chunks
// holding at least one such shell make up 55% and 20%.
//
// The shells come from a table sorted by class (angular momentum, highest
// first, and kind of row map), so that four consecutive entries mostly share
// one: they are evaluated together, one per 16 lanes of a wave.
#pragma once
#include "fused_tile.h"

namespace okmi_fused {

// One list entry: the shell (relative to the list's base index) and its class,
// its first AO row (C column) and its live primitives among the first four,
// its squared distance to the tile's box, and what its evaluation reads (its
// place in the table of row maps among them; from LDS, where a load of the shell's record would be waited for).
struct alignas(16) LiveShell {
    unsigned idcls, rowlive;
    double d2;
    double alpha[4], d[4], c[3];
    int t0;
};
constexpr int LIST_ID_BITS = 18, LIST_ROW_BITS = 29;
constexpr unsigned LIST_ID_MASK = (1u << LIST_ID_BITS) - 1, LIST_ROW_MASK = (1u << LIST_ROW_BITS) - 1;

// population count of the bits of m below this lane
__device__ __forceinline__ int bits_below(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

// Bounding box of the tile's points into sbox (lo x, y, z, hi x, y, z): wave w
// < 3 reduces axis w over its lanes (lane l holds point l of the tile).  Ready
// after the next barrier.
__device__ __forceinline__ void shared_box(int wave, double px, double py, double pz, double* sbox)
{
    if (wave < 3) {
        const double v = wave == 0 ? px : wave == 1 ? py : pz;
        double lo = v, hi = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            lo = fmin(lo, __shfl_xor(lo, o));
            hi = fmax(hi, __shfl_xor(hi, o));
        }
        sbox[wave] = lo;       // (every lane the same value)
        sbox[3 + wave] = hi;
    }
}

// Tests the table's next LCAP shells (from t0; thread i < LCAP takes shell
// t0 + i) against the box and appends those in reach to ent, which holds
// `cnt` entries and has room for LCAP.  Returns the entries added, or -1 if
// they do not fit (nothing is appended).  Called by all NW waves; ent is ready
// after the next barrier.  wsum: NW ints, free again after the next barrier.
template <int LCAP, int NW>
__device__ __forceinline__ int append_live(const ListRec* shells, int nsh, int t0, int base, const double* sbox,
                                           LiveShell* ent, int* wsum, int cnt)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = t0 + (int)threadIdx.x;
    bool hit = false;
    LiveShell e{};
    if ((int)threadIdx.x < LCAP && i < nsh) {
        const ListRec sh = shells[i];
        double d2 = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double d = fmax(fmax(sbox[k] - sh.c[k], sh.c[k] - sbox[3 + k]), 0.0);
            d2 = fma(d, d, d2);
            e.c[k] = sh.c[k];
        }
        hit = d2 < sh.rcut2;
        int live = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            live += d2 < sh.prcut2[q];
            e.alpha[q] = sh.alpha[q];
            e.d[q] = sh.d[q];
        }
        e.d2 = d2;
        e.t0 = sh.t0;
        e.idcls = (unsigned)(i - base) | (unsigned)sh.cls << LIST_ID_BITS;
        e.rowlive = (unsigned)sh.row0 | (unsigned)live << LIST_ROW_BITS;
    }
    const unsigned long long m = __builtin_amdgcn_ballot_w64(hit);
    if (lane == 0) wsum[wave] = __builtin_popcountll(m);
    __syncthreads();
    int n = 0, n0 = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int c = __builtin_amdgcn_readfirstlane(wsum[w]);
        if (w < wave) n0 += c;
        n += c;
    }
    if (cnt + n > LCAP) return -1;
    if (hit) ent[cnt + n0 + bits_below(m)] = e;
    return n;
}

}  // namespace okmi_fused
