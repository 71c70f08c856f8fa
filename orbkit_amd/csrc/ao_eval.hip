// AO evaluation kernel: one lane per grid point, wave-uniform loop over
// shells, output rows written as coalesced SoA  out[set][row][ld].
//
// Replaces orbkit's c_lcreator (orbkit/c_grid-based.c:9-79) looped over
// contractions by cy_core.aocreator (orbkit/cy_core.pyx:49-78), the ORCA row
// renormalisation (orbkit/core.py:98-100) and cartesian2spherical
// (orbkit/core.py:135-176): all of these are one pass here.
#include "okmi_internal.h"
#include "ao_device.h"

#include <type_traits>

namespace {

struct AoArgs {
    const ShellRec* shells;
    const PrimRec* prims;
    const double* T;
    GridDesc grid;
    int64_t p0, np;
    int64_t ld;          // row stride of out (elements)
    int64_t set_stride;  // stride between derivative sets (elements)
    int nshell;
    int need1;                 // first derivatives (radial sum S1) needed
    int dst[OKMI_MAX_SETS];    // output set of derivative code c, -1: not written by this launch
    // brick mode (regular grids): wave w of the launch takes brick bk0 + w
    // (4x4x4 points, z fastest) of the nbx x nby x nbz bricks and writes
    // columns tile_stride w + lane (64: whole rows); lanes of a brick outside the grid repeat its
    // nearest grid point, so every column of the nbk bricks is written
    int brick;
    int64_t bk0, nbk, nbx, nby, nbz, tile_stride;
    // optional live-chunk mask (AoLiveMask): the wave walks only the shells
    // of its tile's live chunks (chunk table and work-ordered shells of the
    // fused layout); null: every shell of `shells`
    const unsigned long long* live_mask;
    int mask_words, mask_shift;
    const int2* chunks;        // per chunk: first work entry, shells | used rows << 16
    const ShellRec* wshells;   // work order, internal rows, fused radii, PrimRec primitives
};

// squared distance from a shell centre to the wave's points' bounding box
// (wave-uniform); lo/hi are wave minima/maxima of the point coordinates
__device__ __forceinline__ double box_dist2(const double (&lo)[3], const double (&hi)[3], const ShellRec& sh)
{
    const double c[3] = {sh.cx, sh.cy, sh.cz};
    double d2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double d = fmax(fmax(lo[k] - c[k], c[k] - hi[k]), 0.0);
        d2 = fma(d, d, d2);
    }
    return d2;
}

// FP64 outputs use the libm-accurate exponential (parity path); FP32
// outputs the reduced one (relative error < 2.6e-9, far below FP32's 6e-8)
template <typename OutT>
__device__ __forceinline__ double gauss_out(double t)
{
    if constexpr (sizeof(OutT) == 8) return gauss_f64(t);
    else return gauss_f64_fast(t);
}

// rows of one shell from its canonical Cartesian values c, stored into the
// AO set starting at o (row stride a.ld)
template <int L, typename OutT>
__device__ __forceinline__ void store_rows(const AoArgs& a, const ShellRec& sh, const double* c, OutT* o, bool act)
{
    constexpr int NC = ncart(L);
    // streaming (non-temporal) stores: the sets are read back by a later
    // kernel from HBM, so the rows are not kept in L2
    auto store = [&](int r, double v) {
        if (act) __builtin_nontemporal_store((OutT)v, &o[(int64_t)r * a.ld]);
    };
    // standard spherical / Cartesian shells: sparse compile-time rows;
    // other transforms (ORCA row factors, custom maps): the dense block
    if (sh.kind == SHELL_T_SPHERICAL) {
        sph_rows_to<L, 0>(c, store);
    } else if (sh.kind == SHELL_T_CARTESIAN) {
        cart_rows_to<L, 0>(c, store);
    } else {
        const OKMI_CONST double* T = cptr(a.T) + sh.t0;
        for (int r = 0; r < sh.nrow; ++r) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < NC; ++k) v = fma(T[r * NC + k], c[k], v);
            store(r, v);
        }
    }
}

// One shell at the lane's point for the derivative codes of group GRP:
// 0 = value and first derivatives (codes 0-3, from shared monomials),
// 1 = second derivatives (codes 4-9, cart_all; the mixed ones with orbkit's
// formula).  Only codes with a destination set are written.
template <int L, int GRP, typename OutT>
__device__ __forceinline__ void shell_out(const AoArgs& a, const ShellRec& sh, double d2, double px, double py,
                                          double pz, int64_t i, bool act, OutT* out)
{
    const double X = px - sh.cx, Y = py - sh.cy, Z = pz - sh.cz;
    const double rr = X * X + Y * Y + Z * Z;
    const bool need1 = GRP == 1 || a.need1;
    double S0 = 0.0, S1 = 0.0, S2 = 0.0;
    for (int p = 0; p < sh.nprim; ++p) {
        const PrimRec pr = load_prim(a.prims, sh.prim0 + p);
        if (d2 >= pr.rcut2) continue;   // below 1e-40 for every point of the wave
        const double de = pr.d * gauss_out<OutT>(pr.alpha * rr);
        S0 += de;
        if (need1) S1 += (-2.0 * pr.alpha) * de;
        if constexpr (GRP == 1) S2 += (4.0 * pr.alpha * pr.alpha) * de;
    }
    ShellPows<L, double> P;
    P.init(X, Y, Z);
    constexpr int NC = ncart(L);
    OutT* o = out + (int64_t)sh.row0 * a.ld + i;
    double c[NC];
    if constexpr (GRP == 0) {
        double m[NC], u[L > 0 ? ncart(L - 1) : 1];
        first_mono<L, 0, double>(P, m);
        if (a.dst[0] >= 0) {
#pragma unroll
            for (int k = 0; k < NC; ++k) c[k] = m[k] * S0;
            store_rows<L, OutT>(a, sh, c, o + a.dst[0] * a.set_stride, act);
        }
        if (!need1) return;
        lower_mono<L, 0, double>(P, S0, u);
        if (a.dst[1] >= 0) {
            first_deriv<L, 0, 0, double>(m, u, X * S1, c);
            store_rows<L, OutT>(a, sh, c, o + a.dst[1] * a.set_stride, act);
        }
        if (a.dst[2] >= 0) {
            first_deriv<L, 1, 0, double>(m, u, Y * S1, c);
            store_rows<L, OutT>(a, sh, c, o + a.dst[2] * a.set_stride, act);
        }
        if (a.dst[3] >= 0) {
            first_deriv<L, 2, 0, double>(m, u, Z * S1, c);
            store_rows<L, OutT>(a, sh, c, o + a.dst[3] * a.set_stride, act);
        }
    } else {
#define OKMI_SECOND(D)                                                             \
        if (a.dst[D] >= 0) {                                                       \
            cart_all<L, D, double>(P, S0, S1, S2, c);                              \
            store_rows<L, OutT>(a, sh, c, o + a.dst[D] * a.set_stride, act);      \
        }
        OKMI_SECOND(4) OKMI_SECOND(5) OKMI_SECOND(6) OKMI_SECOND(7) OKMI_SECOND(8) OKMI_SECOND(9)
#undef OKMI_SECOND
    }
}

// Second derivatives of live chunks (group 1), and every set of a basis with a
// shell of more than 32 rows, which has no list tables.  Occupancy (waves/SIMD)
// the register allocation targets without spilling: FP32 output 4 (group 0) and 3
// (group 1), FP64 output 3 and 2
template <typename OutT, int GRP>
__global__ __launch_bounds__(256, sizeof(OutT) == 4 ? (GRP == 0 ? 4 : 3) : (GRP == 0 ? 3 : 2))
void k_ao_eval(AoArgs a, OutT* __restrict__ out)
{
    int64_t i;
    bool act;
    double px, py, pz;
    if (a.brick) {
        const GridDesc& g = a.grid;
        const int lane = threadIdx.x & 63;
        const int64_t wb = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
        int64_t t = a.bk0 + wb;
        const int64_t bz = t % a.nbz;
        t /= a.nbz;
        const int64_t by = t % a.nby, bx = t / a.nby;
        int64_t ix = 4 * bx + (lane >> 4), iy = 4 * by + ((lane >> 2) & 3), iz = 4 * bz + (lane & 3);
        ix = ix < g.nx ? ix : g.nx - 1;
        iy = iy < g.ny ? iy : g.ny - 1;
        iz = iz < g.nz ? iz : g.nz - 1;
        act = wb < a.nbk;
        i = wb * a.tile_stride + lane;
        px = g.x[ix]; py = g.y[iy]; pz = g.z[iz];
    } else {
        i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        act = i < a.np;
        grid_point(a.grid, a.p0 + (act ? i : 0), px, py, pz);
    }
    // bounding box of the wave's points (inactive lanes repeat point 0,
    // which only enlarges the box)
    double lo[3] = {px, py, pz}, hi[3] = {px, py, pz};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fmin(lo[k], __shfl_xor(lo[k], o));
            hi[k] = fmax(hi[k], __shfl_xor(hi[k], o));
        }
    // one shell for the wave's points: its rows evaluated, or zero when it is
    // out of reach (every value and derivative below the screening bound)
    auto shell = [&](const ShellRec& sh) {
        const double d2 = uniform(box_dist2(lo, hi, sh));
        if (d2 >= sh.rcut2) {
            if (act)
                for (int c = 0; c < OKMI_MAX_SETS; ++c) {
                    if (a.dst[c] < 0) continue;
                    OutT* o = out + a.dst[c] * a.set_stride + (int64_t)sh.row0 * a.ld + i;
                    for (int r = 0; r < sh.nrow; ++r) __builtin_nontemporal_store((OutT)0, &o[(int64_t)r * a.ld]);
                }
            return;
        }
        switch (sh.l) {
        case 0: shell_out<0, GRP, OutT>(a, sh, d2, px, py, pz, i, act, out); break;
        case 1: shell_out<1, GRP, OutT>(a, sh, d2, px, py, pz, i, act, out); break;
        case 2: shell_out<2, GRP, OutT>(a, sh, d2, px, py, pz, i, act, out); break;
        case 3: shell_out<3, GRP, OutT>(a, sh, d2, px, py, pz, i, act, out); break;
        default: shell_out<4, GRP, OutT>(a, sh, d2, px, py, pz, i, act, out); break;
        }
    };
    if (!a.live_mask) {
        for (int s = 0; s < a.nshell; ++s) shell(load_shell(a.shells, s));
        return;
    }
    // the shells of the live chunks of this wave's tile; the rows of the
    // other chunks are never read, and are left unwritten.  Masks exist for
    // the tiles holding the launch's points only: a wave past the last point
    // (the grid's rounding) has nothing to write and stops here.
    const int64_t wv = a.brick ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)
                               : ((int64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63)) >> 6;
    if (a.brick ? wv >= a.nbk : wv * 64 >= a.np) return;
    const int64_t wt = wv >> a.mask_shift;
    const unsigned long long* mrow = a.live_mask + wt * a.mask_words;
    for (int w = 0; w < a.mask_words; ++w) {
        const unsigned long long m0 = mrow[w];
        unsigned long long m = ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(m0 >> 32)) << 32) |
                               (unsigned)__builtin_amdgcn_readfirstlane((unsigned)m0);
        while (m) {
            const int c = 64 * w + __builtin_ctzll(m);
            m &= m - 1;
            const int2 cw = load_int2(a.chunks, c);
            const int nsh = cw.y & 0xffff;
            for (int e = 0; e < nsh; ++e) shell(load_shell(a.wshells, cw.x + e));
        }
    }
}

// Values of every shell (codes of PASS: 0 value, 1 value and first
// derivatives, 2 and 3 value and diagonal or mixed second ones), one lane per
// point.  The four waves of a workgroup take the same 64 points and every
// fourth shell each (blockIdx.y: a part of the shells, where the points alone
// would leave the chip short of waves), so that the waves in flight cover the
// scalar load of a shell's record, which holds its first four primitives.
// Bound by its stores (3.35 GB in 608 us, 5.5 TB/s, against 6.9 of a fill).  They
// go through L2: a row of an odd number of points begins inside a line, whose
// two parts two waves write, and non-temporal stores sent the parts to memory one
// by one (126,362 points x 162 rows: 68 us non-temporal, 42 through L2; rows of
// whole lines, 400 x 4 x 261,568: 631 and 608 us).  The parts meet there only if
// neighbouring tiles run on one XCD: workgroups are dealt to the eight XCDs in
// turn, so each XCD takes one eighth of the tiles in order (1,200 rows, tiles
// in turn and in eighths: 3 sets of 60,001 points 648 and 544 us, 4 sets of
// 91,125 points 1,427 and 1,140 us; 1 set of 262,144, whole lines, 477 and 480 us).
// FP32 (exponential of gauss_out): 1,200 rows x 3 sets of 91,125 points 469 us,
// of 262,144 points 713 us (k_ao_eval, one wave per tile and non-temporal
// stores: 715 and 843).
struct AoListArgs {
    const ListRec* shells;      // by class, output rows, radii of OKMI_SCREEN
    const PrimGroup* more;
    const double* T;
    GridDesc grid;
    int64_t p0, np, ld, set_stride;
    int nsh, per;               // shells; per blockIdx.y
    int dst[4];                 // output set of the pass's AO sets, -1: not wanted
};

template <int PASS> struct AoSets { static constexpr int n = PASS == 0 ? 1 : 4; };

template <int L, bool SPH, int PASS, typename OutT>
__device__ __forceinline__ void ao_rows(const AoListArgs& a, OutT* o, bool act, double X, double Y, double Z, double S0,
                                        double S1, double S2)
{
    constexpr int NS = AoSets<PASS>::n;
    each_row<0>(RowSets<L, SPH, PASS>(X, Y, Z, S0, S1, S2), [&](int r, const double (&v)[NS]) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
            if (a.dst[s] >= 0 && act) o[a.dst[s] * a.set_stride + r * a.ld] = (OutT)v[s];
    });
}

template <int L, int PASS, typename OutT>
__device__ __forceinline__ void ao_general(const AoListArgs& a, const ListRec& sh, OutT* o, bool act, double X, double Y,
                                           double Z, double S0, double S1, double S2)
{
    constexpr int NS = AoSets<PASS>::n, NC = ncart(L);
    constexpr int c1 = PASS == 1 ? 1 : PASS == 2 ? 4 : 7;
    ShellPows<L, double> P;
    P.init(X, Y, Z);
    const OKMI_CONST double* T = cptr(a.T) + sh.t0;
    auto set = [&](auto code, int s) {
        if (a.dst[s] < 0) return;
        double c[NC];
        cart_all<L, decltype(code)::value, double>(P, S0, S1, S2, c);
        for (int r = 0; r < sh.nrow; ++r) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < NC; ++k) v = fma(T[r * NC + k], c[k], v);
            if (act) o[a.dst[s] * a.set_stride + r * a.ld] = (OutT)v;
        }
    };
    set(std::integral_constant<int, 0>{}, 0);
    if constexpr (NS > 1) {
        set(std::integral_constant<int, c1>{}, 1);
        set(std::integral_constant<int, c1 + 1>{}, 2);
        set(std::integral_constant<int, c1 + 2>{}, 3);
    }
}

// squared distance from a record's centre to the box (wave-uniform)
__device__ __forceinline__ double list_dist2(const double (&lo)[3], const double (&hi)[3], const ListRec& sh)
{
    double d2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double d = fmax(fmax(lo[k] - sh.c[k], sh.c[k] - hi[k]), 0.0);
        d2 = fma(d, d, d2);
    }
    return uniform(d2);
}

// the rows of one shell in reach (squared distance d2 to the wave's box) at
// the lane's point, its first row's place at o
template <int PASS, typename OutT>
__device__ __forceinline__ void list_shell(const AoListArgs& a, const ListRec& sh, double d2, double px, double py, double pz,
                                           OutT* o, bool act)
{
    constexpr bool need1 = PASS == 1 || PASS == 2, need2 = PASS >= 2;
    const double X = px - sh.c[0], Y = py - sh.c[1], Z = pz - sh.c[2];
    const double rr = X * X + Y * Y + Z * Z;
    double S0 = 0.0, S1 = 0.0, S2 = 0.0;
    auto prim = [&](double alpha, double d) {
        const double de = d * gauss_out<OutT>(alpha * rr);
        S0 += de;
        if constexpr (need1) S1 = fma(alpha, de, S1);
        if constexpr (need2) S2 = fma(alpha * alpha, de, S2);
    };
    // the primitives in reach lead (radii descend)
    if (d2 < sh.prcut2[0]) prim(sh.alpha[0], sh.d[0]);
    if (d2 < sh.prcut2[1]) prim(sh.alpha[1], sh.d[1]);
    if (d2 < sh.prcut2[2]) prim(sh.alpha[2], sh.d[2]);
    if (d2 < sh.prcut2[3]) {
        prim(sh.alpha[3], sh.d[3]);
        for (int q = 4; q < sh.nprim; ++q) {
            const OKMI_CONST PrimGroup* g = cptr(a.more) + sh.more + ((q - 4) >> 2);
            if (!(d2 < g->rcut2[q & 3])) break;
            prim(g->alpha[q & 3], g->d[q & 3]);
        }
    }
    S1 *= -2.0;
    S2 *= 4.0;
#define OKMI_AO_CASE(L)                                                                              \
    case L:                                                                                          \
        if (sh.kind == SHELL_T_GENERAL) ao_general<L, PASS>(a, sh, o, act, X, Y, Z, S0, S1, S2);     \
        else if (L <= 3 && sh.kind == SHELL_T_SPHERICAL)                                             \
            ao_rows<(L <= 3 ? L : 0), true, PASS>(a, o, act, X, Y, Z, S0, S1, S2);                   \
        else ao_rows<L, false, PASS>(a, o, act, X, Y, Z, S0, S1, S2);                                \
        break;
    switch (sh.l) {
        OKMI_AO_CASE(0) OKMI_AO_CASE(1) OKMI_AO_CASE(2) OKMI_AO_CASE(3)
    default:
        OKMI_AO_CASE(4)
    }
#undef OKMI_AO_CASE
}

template <int PASS, typename OutT>
__global__ __launch_bounds__(256, PASS == 0 ? 4 : 3) void k_ao_list(AoListArgs a, OutT* __restrict__ out)
{
    constexpr int NS = AoSets<PASS>::n;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned xcd = blockIdx.x & 7, eighth = gridDim.x >> 3, rest = gridDim.x & 7;
    const unsigned tile = xcd * eighth + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
    const int64_t i = (int64_t)tile * 64 + lane;
    const bool act = i < a.np;
    double px, py, pz;
    grid_point(a.grid, a.p0 + (act ? i : a.np - 1), px, py, pz);
    double lo[3] = {px, py, pz}, hi[3] = {px, py, pz};   // the wave's bounding box
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fmin(lo[k], __shfl_xor(lo[k], o));
            hi[k] = fmax(hi[k], __shfl_xor(hi[k], o));
        }
    const int end = min(a.nsh, ((int)blockIdx.y + 1) * a.per);
    for (int s = (int)blockIdx.y * a.per + wave; s < end; s += 4) {
        const ListRec sh = load_list(a.shells, s);
        const double d2 = list_dist2(lo, hi, sh);
        OutT* o = out + sh.row0 * a.ld + i;
        if (!(d2 < sh.rcut2)) {   // every value and derivative below the screening bound
            if (act)
                for (int q = 0; q < NS; ++q) {
                    if (a.dst[q] < 0) continue;
                    for (int r = 0; r < sh.nrow; ++r) o[a.dst[q] * a.set_stride + r * a.ld] = (OutT)0;
                }
            continue;
        }
        list_shell<PASS>(a, sh, d2, px, py, pz, o, act);
    }
}

// Values and first derivatives (PASS 0, 1) of the shells in a tile's live chunks
// (AoLiveMask), the AO sets of the staged contractions.  The four waves of a
// workgroup take the same 64 points and every fourth of those shells: with one
// wave per tile and one scalar load per primitive (each waited for in turn), a
// pass of 3,277 tiles left the chip a single, latency-bound round of waves.
// Per pass of 209,664 points x 4 FP32 sets (2,950 AOs): 393 -> 212 us; 512,000
// points x 1 set (400 AOs): FP64 211 -> 141 us, FP32 152 -> 73 us.
struct AoLiveArgs {
    AoListArgs l;               // shells: work order, internal rows
    const int2* chunks;         // per chunk: first shell, shells | used rows << 16
    const unsigned long long* mask;
    int words, shift, quads;    // as AoLiveMask
    int brick;                  // as AoArgs
    int64_t bk0, nbx, nby, nbz, tile_stride;
};

template <int PASS, typename OutT>
__global__ __launch_bounds__(256, PASS == 0 ? 4 : 3) void k_ao_live(AoLiveArgs a, OutT* __restrict__ out)
{
    constexpr int NS = AoSets<PASS>::n;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t tile = blockIdx.x;
    bool act = true;
    double px, py, pz;
    if (a.brick) {   // lanes outside the grid repeat its nearest point
        const GridDesc& g = a.l.grid;
        unsigned t = (unsigned)(a.bk0 + tile);   // (2^32 bricks would be 2 TB of densities)
        const unsigned nbz = (unsigned)a.nbz, nby = (unsigned)a.nby;
        const int64_t bz = t % nbz;
        t /= nbz;
        const int64_t by = t % nby, bx = t / nby;
        const int64_t ix = min(4 * bx + (lane >> 4), g.nx - 1), iy = min(4 * by + ((lane >> 2) & 3), g.ny - 1);
        const int64_t iz = min(4 * bz + (lane & 3), g.nz - 1);
        px = g.x[ix]; py = g.y[iy]; pz = g.z[iz];
    } else {   // (lanes past the end repeat the first point)
        const int64_t i = tile * 64 + lane;
        act = i < a.l.np;
        grid_point(a.l.grid, a.l.p0 + (act ? i : 0), px, py, pz);
    }
    double lo[3] = {px, py, pz}, hi[3] = {px, py, pz};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fmin(lo[k], __shfl_xor(lo[k], o));
            hi[k] = fmax(hi[k], __shfl_xor(hi[k], o));
        }
    OutT* base = out + tile * a.tile_stride + lane;
    const unsigned long long* mrow = a.mask + (tile >> a.shift) * a.words;
    int skip = wave;   // shells until this wave's next one
    for (int w = 0; w < a.words; ++w) {
        const unsigned long long m0 = mrow[w];
        unsigned long long m = ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(m0 >> 32)) << 32) |
                               (unsigned)__builtin_amdgcn_readfirstlane((unsigned)m0);
        while (m) {
            const int bit = __builtin_ctzll(m);
            int c = 64 * w + bit;
            unsigned quads = 0xff;   // the chunk's quads that are read
            if (a.quads) {
                c >>= 3;
                quads = (unsigned)(m >> (bit & ~7)) & 0xff;
                m &= ~(0xffull << (bit & ~7));
            } else {
                m &= m - 1;
            }
            const int2 cw = load_int2(a.chunks, c);
            const int nsh = cw.y & 0xffff;
            for (; skip < nsh; skip += 4) {
                const ListRec sh = load_list(a.l.shells, cw.x + skip);
                const double d2 = list_dist2(lo, hi, sh);
                OutT* o = base + sh.row0 * a.l.ld;
                if (d2 < sh.rcut2) {
                    list_shell<PASS>(a.l, sh, d2, px, py, pz, o, act);
                } else if (act) {   // out of the wave's reach: zero rows
                    for (int q = 0; q < NS; ++q) {
                        if (a.l.dst[q] < 0) continue;
                        for (int r = 0; r < sh.nrow; ++r)
                            if (quads >> (((sh.row0 + r) & 31) >> 2) & 1)
                                o[a.l.dst[q] * a.l.set_stride + r * a.l.ld] = (OutT)0;
                    }
                }
            }
            skip -= nsh;
        }
    }
}

// Waves that fill the chip several times over: the shells are split into parts
// until the points give as many (small grids).
constexpr int64_t AO_WAVES = 16384;

template <typename OutT>
void launch_ao_list(const OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, const int (&first)[OKMI_MAX_SETS],
                    OutT* out, int64_t ld, int64_t set_stride, hipStream_t st)
{
    AoListArgs a{};
    a.shells = b->d_lshells_a;
    a.more = b->d_lgroups_a;
    a.T = b->d_T;
    a.grid = g;
    a.ld = ld;
    a.set_stride = set_stride;
    a.nsh = b->nshell;
    const int64_t blocks = (np + 63) / 64;
    // (at least two shells per wave)
    const int64_t parts = std::max<int64_t>(1, std::min<int64_t>((AO_WAVES / 4 + blocks - 1) / blocks, b->nshell / 8));
    a.per = (int)((b->nshell + parts - 1) / parts);
    const dim3 blk(256);
    auto launch = [&](auto pass) {
        for (int64_t t = 0; t < blocks; t += OKMI_MAX_BLOCKS) {
            a.p0 = p0 + 64 * t;
            a.np = std::min(np - 64 * t, 64 * OKMI_MAX_BLOCKS);
            const dim3 grd((unsigned)((a.np + 63) / 64), (unsigned)((b->nshell + a.per - 1) / a.per));
            hipLaunchKernelGGL((k_ao_list<decltype(pass)::value, OutT>), grd, blk, 0, st, a, out + 64 * t);
        }
    };
    bool value = first[0] >= 0;   // written by the first pass launched
    auto pass = [&](int c1) {     // codes c1 .. c1 + 2
        bool any = false;
        for (int q = 0; q < 3; ++q) {
            a.dst[1 + q] = first[c1 + q];
            any = any || first[c1 + q] >= 0;
        }
        if (!any) return false;
        a.dst[0] = value ? first[0] : -1;
        value = false;
        return true;
    };
    if (pass(1)) launch(std::integral_constant<int, 1>{});
    if (pass(4)) launch(std::integral_constant<int, 2>{});
    if (pass(7)) launch(std::integral_constant<int, 3>{});
    if (value) {
        a.dst[0] = first[0];
        launch(std::integral_constant<int, 0>{});
    }
}

}  // namespace

int okmi_launch_ao_eval(const OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, const int* drv, int ndrv,
                        int out_dtype, void* out, int64_t ld, int64_t set_stride, hipStream_t st)
{
    return okmi_launch_ao_eval_ex(b, b->d_shells, b->d_prims, g, p0, np, nullptr, drv, ndrv, out_dtype, out, ld,
                                  set_stride, st);
}

int okmi_launch_ao_eval_ex(const OkmiBasis* b, const ShellRec* shells, const PrimRec* prims, const GridDesc& g,
                           int64_t p0, int64_t np, const AoBricks* bricks, const int* drv, int ndrv, int out_dtype,
                           void* out, int64_t ld, int64_t set_stride, hipStream_t st, const AoLiveMask* live)
{
    if (np <= 0 && !bricks) return 0;
    AoArgs a{};
    if (live) {
        a.live_mask = live->mask;
        a.mask_words = live->words;
        a.mask_shift = live->shift;
        a.chunks = b->d_chunks;
        a.wshells = live->wshells ? live->wshells : b->d_wshells;
    }
    a.shells = shells;
    a.prims = prims;
    a.T = b->d_T;
    a.grid = g;
    a.p0 = p0;
    a.np = np;
    a.ld = ld;
    a.set_stride = set_stride;
    a.nshell = b->nshell;
    a.tile_stride = live ? live->tile_stride : 64;
    // each code's first set; the groups write those, repeats are copies
    int first[OKMI_MAX_SETS];
    for (int c = 0; c < OKMI_MAX_SETS; ++c) first[c] = -1;
    for (int j = 0; j < ndrv; ++j) {
        if (drv[j] < 0 || drv[j] >= OKMI_MAX_SETS) {
            okmi_set_error("ao_eval: derivative code %d is not in 0..9", drv[j]);
            return 1;
        }
        if (first[drv[j]] < 0) first[drv[j]] = j;
    }
    dim3 blk(256), grd((unsigned)((np + 255) / 256));
    int64_t width = np;   // columns written per row
    if (bricks) {
        if (bricks->nbk <= 0) return 0;
        a.brick = 1;
        a.bk0 = bricks->bk0; a.nbk = bricks->nbk;
        a.tile_stride = bricks->tile_stride;
        a.nbx = bricks->nbx; a.nby = bricks->nby; a.nbz = bricks->nbz;
        grd = dim3((unsigned)((bricks->nbk + 3) / 4));
        width = bricks->nbk * 64;
    }
    OkmiProfScope prof("ao_eval", st);
    const bool list = !bricks && !live && shells == b->d_shells && b->d_lshells_a;
    if (list && out_dtype == OKMI_F64) launch_ao_list(b, g, p0, np, first, (double*)out, ld, set_stride, st);
    else if (list) launch_ao_list(b, g, p0, np, first, (float*)out, ld, set_stride, st);
    // values and first derivatives of live chunks (second derivatives: k_ao_eval's group 1)
    if (live) {
        AoLiveArgs w{};
        const bool split = live->wshells && live->wshells == b->d_wshells_s;
        w.l.shells = split ? b->d_wlist_s : b->d_wlist;
        w.l.more = split ? b->d_wlist_groups_s : b->d_wlist_groups;
        w.l.T = b->d_T;
        w.l.grid = g; w.l.p0 = p0; w.l.np = np; w.l.ld = ld; w.l.set_stride = set_stride;
        for (int c = 0; c < 4; ++c) w.l.dst[c] = first[c];
        w.chunks = b->d_chunks;
        w.mask = live->mask; w.words = live->words; w.shift = live->shift; w.quads = live->quads;
        w.brick = a.brick; w.bk0 = a.bk0; w.nbx = a.nbx; w.nby = a.nby; w.nbz = a.nbz; w.tile_stride = a.tile_stride;
        const dim3 tiles((unsigned)(bricks ? bricks->nbk : (np + 63) / 64));
        const bool first_deriv = first[1] >= 0 || first[2] >= 0 || first[3] >= 0;
        if (out_dtype == OKMI_F64) {
            if (first_deriv) hipLaunchKernelGGL((k_ao_live<1, double>), tiles, blk, 0, st, w, (double*)out);
            else if (first[0] >= 0) hipLaunchKernelGGL((k_ao_live<0, double>), tiles, blk, 0, st, w, (double*)out);
        } else {
            if (first_deriv) hipLaunchKernelGGL((k_ao_live<1, float>), tiles, blk, 0, st, w, (float*)out);
            else if (first[0] >= 0) hipLaunchKernelGGL((k_ao_live<0, float>), tiles, blk, 0, st, w, (float*)out);
        }
    }
    for (int grp = live ? 1 : 0; grp < 2 && !list; ++grp) {
        const int c0 = grp == 0 ? 0 : 4, c1 = grp == 0 ? 4 : OKMI_MAX_SETS;
        bool any = false;
        for (int c = 0; c < OKMI_MAX_SETS; ++c) {
            a.dst[c] = c >= c0 && c < c1 ? first[c] : -1;
            any |= a.dst[c] >= 0;
        }
        if (!any) continue;
        a.need1 = first[1] >= 0 || first[2] >= 0 || first[3] >= 0;
        if (out_dtype == OKMI_F64) {
            if (grp == 0) hipLaunchKernelGGL((k_ao_eval<double, 0>), grd, blk, 0, st, a, (double*)out);
            else hipLaunchKernelGGL((k_ao_eval<double, 1>), grd, blk, 0, st, a, (double*)out);
        } else {
            if (grp == 0) hipLaunchKernelGGL((k_ao_eval<float, 0>), grd, blk, 0, st, a, (float*)out);
            else hipLaunchKernelGGL((k_ao_eval<float, 1>), grd, blk, 0, st, a, (float*)out);
        }
    }
    const size_t es = out_dtype == OKMI_F64 ? sizeof(double) : sizeof(float);
    for (int j = 0; j < ndrv; ++j) {
        const int f = first[drv[j]];
        if (f == j) continue;
        char* base = (char*)out;
        const hipError_t e = hipMemcpy2DAsync(base + (size_t)j * set_stride * es, (size_t)ld * es,
                                              base + (size_t)f * set_stride * es, (size_t)ld * es, (size_t)width * es,
                                              (size_t)b->nao, hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) return okmi_hip_fail(e, "ao_eval: repeated derivative set");
    }
    return okmi_check_launch("ao_eval");
}
