// Per-tile lists of the shells in reach, for the FP64 kernels that contract
// only those: a 64-point brick reaches about a quarter of the AO rows of a
// 20-atom molecule and 7% of those of 200 atoms, where fixed 32-row chunks
// holding at least one such shell make up 55% and 20%.
//
// The shells are taken from a table sorted by angular momentum (highest
// first), so that the shells of one chunk cost about the same and the four
// waves that share a chunk finish together.
#pragma once
#include "fused_tile.h"

namespace okmi_fused {

// One list entry: x = shell (relative to the list's base index) and the
// number of AO rows before it, y = its first AO row (C column).  The entry
// after the last holds the total row count.
constexpr int LIST_ID_BITS = 18;
constexpr unsigned LIST_ID_MASK = (1u << LIST_ID_BITS) - 1;

// value of the previous lanes' bits: population count of m below this lane
__device__ __forceinline__ int bits_below(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

// Tests the table's next BLK shells (from t0; thread i < BLK takes shell
// t0 + i) against the box and appends those in reach to ent, which holds
// `cnt` entries and `rows` rows so far and has room for LCAP.  Returns the
// entries added, or -1 if they do not fit (nothing is appended).  Called by
// all 256 threads; ent is ready after the next barrier.  wsum: 8 ints, free
// again after the next barrier.
template <int LCAP, int BLK>
__device__ __forceinline__ int append_live(const ShellRec* shells, int nsh, int t0, int base, const Box& box,
                                           uint2* ent, int* wsum, int cnt, int& rows)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = t0 + (int)threadIdx.x;
    int nrow = 0, row0 = 0;
    if ((int)threadIdx.x < BLK && i < nsh) {
        const ShellRec sh = shells[i];
        row0 = sh.row0;
        if (box.dist2(sh) < sh.rcut2) nrow = sh.nrow;
    }
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(nrow > 0);
    int before = 0, total = 0;   // rows of the wave's live shells before this lane, and in all
#pragma unroll
    for (int b = 0; b < 6; ++b) {   // nrow <= 32
        const unsigned long long m = __builtin_amdgcn_ballot_w64((nrow >> b & 1) != 0);
        before += bits_below(m) << b;
        total += __builtin_popcountll(m) << b;
    }
    if (lane == 0) {
        wsum[2 * wave] = __builtin_popcountll(hit);
        wsum[2 * wave + 1] = total;
    }
    __syncthreads();
    int n = 0, nr = 0, n0 = 0, r0 = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        if (w == wave) {
            n0 = n;
            r0 = nr;
        }
        n += wsum[2 * w];
        nr += wsum[2 * w + 1];
    }
    n = __builtin_amdgcn_readfirstlane(n);
    nr = __builtin_amdgcn_readfirstlane(nr);
    if (cnt + n > LCAP) return -1;
    if (nrow > 0)
        ent[cnt + n0 + bits_below(hit)] =
            uint2{(unsigned)(i - base) | (unsigned)(rows + r0 + before) << LIST_ID_BITS, (unsigned)row0};
    rows += nr;
    if (threadIdx.x == 0) ent[cnt + n].x = (unsigned)rows << LIST_ID_BITS;
    return n;
}

// The next chunk of a list: entries s .. s + n - 1, whole shells of at most
// KR rows in all.  Lane j holds entry s + j (ex, ey).
struct ListChunk {
    unsigned ex, ey;
    int n, r0, used;   // entries, the first one's row, rows

    template <int KR>
    __device__ __forceinline__ void next(const uint2* ent, int s, int cnt, int lane)
    {
        const uint2 v = ent[min(s + lane, cnt)];
        ex = v.x;
        ey = v.y;
        const unsigned after = ent[min(s + 1 + lane, cnt)].x >> LIST_ID_BITS;
        r0 = __builtin_amdgcn_readfirstlane(ex >> LIST_ID_BITS);
        const unsigned long long fit = __builtin_amdgcn_ballot_w64(s + lane < cnt && (int)after - r0 <= KR);
        n = __builtin_popcountll(fit);
        used = n > 0 ? (int)__builtin_amdgcn_readlane(after, n - 1) - r0 : 0;
    }
    __device__ __forceinline__ int shell(int j) const { return __builtin_amdgcn_readlane(ex, j) & LIST_ID_MASK; }
    __device__ __forceinline__ int row(int j) const
    {
        return (int)((unsigned)__builtin_amdgcn_readlane(ex, j) >> LIST_ID_BITS) - r0;
    }
    // C column of each row of the chunk, written by one wave
    __device__ __forceinline__ void columns(int* col, int lane) const
    {
        const int first = (int)(ex >> LIST_ID_BITS) - r0;
        // rows of this lane's shell: up to the next lane's first row
        const int last = __shfl_down((int)(ex >> LIST_ID_BITS), 1) - r0;
        if (lane < n)
            for (int r = first; r < (lane == n - 1 ? used : last); ++r) col[r] = (int)ey + r - first;
    }
};

}  // namespace okmi_fused
