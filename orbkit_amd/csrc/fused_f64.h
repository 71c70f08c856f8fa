// FP64 fused kernel: AO values evaluated in FP64 in the registers that the FP64
// matrix cores read them from, contracted with the FP64 MO coefficients; the
// epilogue forms the density terms or stores the MO values.  AO values and (for
// a density) MO values never reach memory.  Compiled with the FP64 MFMAs in the
// VGPR form (no accumulator copies to AGPRs around each MFMA).
//
// FP64 MFMAs and FP64 VALU instructions share one FP64 throughput on gfx950 (a
// CU running MFMA waves and FP64-FMA waves side by side takes the sum of their
// times, 3.56 + 1.10 -> 4.56 ms in a probe), so what pays is less FP64 work and
// nothing that leaves the pipe idle:
//   * MOs are padded to 4, not 16: full 16-MO tiles run on
//     v_mfma_f64_16x16x4f64, the 4-MO groups left over on
//     v_mfma_f64_4x4x4f64 (4 blocks), which has the same rate per flop (68
//     against 72 TFLOP/s measured) and the same B operand layout;
//   * only the shells in reach of the tile are evaluated and contracted
//     (live_shells.h);
//   * four shells of one class are evaluated together, shell g of the four by
//     lanes 16 g .. 16 g + 15 at the wave's 16 points.  Row r of the four is then
//     the B operand of one K step as it stands (lane = k, point), so no AO value
//     passes through LDS and a wave meets no barrier once its tile's list is
//     there.  With the AO tile in LDS (four waves evaluating 20 or 32 rows
//     for 64 points, barrier, contraction, barrier) the pipe stood idle 29% of
//     the time.
//
// A workgroup of four waves owns a tile of 64 points and lists its shells; each
// wave then takes 16 points through the list on its own, the C operands of a
// K step loaded from L2 while the step before it runs.
//
// 4x4x4 lane layout (checked on the GPU with one-hot operands): block
// b = (lane % 16) / 4; A lane 16 k + 4 b + i holds A_b[i][k], B lane
// 16 k + 4 b + j holds B_b[k][j], D lane 16 i + 4 b + j holds D_b[i][j].
// With block b = point group (points 4 b .. 4 b + 3 of the column), i = MO
// and k = AO row, B lane l is AO row k0 + l / 16 at point l % 16 (the
// 16x16x4 B operand) and D lane l is MO m0 + l / 16 at point l % 16.
#pragma once
#include "live_shells.h"

namespace okmi_fused {

// Accumulators of a wave: element i of t[j][s] is MO 16 j + 4 i + lane / 16 and
// r[j][s] MO 16 NT + 4 j + lane / 16 (from the wave's first MO) at point lane % 16,
// AO set s
template <int NT, int NR, int NS> struct MoAcc {
    d4 t[NT > 0 ? NT : 1][NS];
    double r[NR > 0 ? NR : 1][NS];
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
#pragma unroll
            for (int j = 0; j < NT; ++j) t[j][s] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int j = 0; j < NR; ++j) r[j][s] = 0.0;
        }
    }
    // group u of 4 MOs
    __device__ __forceinline__ double get(int u, int s) const { return u < 4 * NT ? t[u / 4][s][u % 4] : r[u - 4 * NT][s]; }
};

// The tile's place: first point of its brick (or of its run of 64 points)
struct TileWhere {
    int x0, y0, z0;   // brick origin (grid indices)
    int64_t first;    // flattened index of the brick's origin, or of the run's first point (relative to p0)

    __device__ __forceinline__ TileWhere(const F64Args& a, unsigned tile)
    {
        const unsigned r = a.dz.div(tile), bx = a.dy.div(r);
        x0 = 4 * (int)bx;
        y0 = 4 * (int)(r - bx * a.dy.d);
        z0 = 4 * (int)(tile - r * a.dz.d);
        first = a.brick ? ((int64_t)x0 * a.grid.ny + y0) * a.grid.nz + z0 : (int64_t)tile * PTS;
    }
    // output index of the tile's point l (relative to p0); false: past the grid's faces or the last point
    __device__ __forceinline__ bool index(const F64Args& a, int l, int64_t& p) const
    {
        if (!a.brick) {
            p = first + l;
            return p < a.np;
        }
        const int dx = l >> 4, dy = l >> 2 & 3, dz = l & 3;
        p = first + (dx * a.grid.ny + dy) * a.grid.nz + dz;
        return x0 + dx < a.grid.nx && y0 + dy < a.grid.ny && z0 + dz < a.grid.nz;
    }
    // its coordinates (those of the nearest point inside where it is past the end)
    __device__ __forceinline__ void point(const F64Args& a, int l, double& px, double& py, double& pz) const
    {
        if (a.brick) {
            px = a.grid.x[min((int64_t)x0 + (l >> 4), a.grid.nx - 1)];
            py = a.grid.y[min((int64_t)y0 + (l >> 2 & 3), a.grid.ny - 1)];
            pz = a.grid.z[min((int64_t)z0 + (l & 3), a.grid.nz - 1)];
        } else {
            grid_point(a.grid, a.p0 + min(first + l, a.np - 1), px, py, pz);
        }
    }
};

// The U groups of 4 MOs of a launch
template <int PASS, int U, bool STD> struct MoSplit {
    static constexpr int NW = 4;                  // waves
    static constexpr int MP = 4 * U;              // padded MO count
    static constexpr int NT = U / 4, NR = U % 4;  // 16-MO and 4-MO accumulators per AO set
    static constexpr int NS = PassCodes<PASS>::n;
    using Acc = MoAcc<NT, NR, NS>;
    // waves per SIMD: the accumulators take 2 U NS registers, the evaluation
    // and the operands in flight about 80
    static constexpr int OCC = !STD ? 2 : 2 * U * NS <= 40 ? 4 : 2 * U * NS <= 80 ? 3 : 2;
    static constexpr int LCAP = 256;              // list entries held at a time
};

// The C operands of one K step: row k = lane / 16 of the four, MOs 16 j +
// lane % 16 (t) and 16 NT + 4 j + lane % 4 (r)
template <int NT, int NR> struct COps {
    double t[NT > 0 ? NT : 1], r[NR > 0 ? NR : 1];
};

// Where they are: C[m][row] as the caller gave it (row stride 1, MO stride
// nao; MOs past the last read the last one, which weighs nothing) or its
// transpose [row][MP]
template <int NT, int NR> struct CWhere {
    typedef const __attribute__((address_space(1))) char gchar;
    typedef const __attribute__((address_space(1))) double gdouble;
    gchar* base;
    unsigned ms, rs;                 // byte strides of an MO and a row (uniform)
    unsigned mt, mtl, mr, mrl;       // lane's MO offset in a tile, the last tile, a group, the last group
    unsigned vt, vtl, vr, vrl;       // the same with the row of the lane's shell

    __device__ __forceinline__ CWhere(const F64Args& a, int mp, int n16)
    {
        base = (gchar*)(a.ct ? a.ct : a.C);
        ms = a.ct ? 8 : 8 * a.nao;
        rs = a.ct ? 8 * a.ct_ld : 8;
        const int last = (a.ct ? mp : a.nmo) - 1;
        mt = n16 * ms;
        mtl = NR == 0 ? last_tile_mo(n16, last, NT) * ms : mt;
        mr = (n16 & 3) * ms;
        mrl = last_group_mo(n16 & 3, last, NT, NR) * ms;
    }
    __device__ __forceinline__ void shell(unsigned row0)
    {
        const unsigned o = row0 * rs;
        vt = mt + o;
        vtl = mtl + o;
        vr = mr + o;
        vrl = mrl + o;
    }
    // row r of the lane's shell
    __device__ __forceinline__ void load(int r, COps<NT, NR>& c) const
    {
        gchar* p = base + (uint64_t)r * rs;
#pragma unroll
        for (int j = 0; j < NT; ++j)
            c.t[j] = *(gdouble*)(p + (uint64_t)(16 * j) * ms + (NR == 0 && j == NT - 1 ? vtl : vt));
#pragma unroll
        for (int j = 0; j < NR; ++j)
            c.r[j] = *(gdouble*)(p + (uint64_t)(16 * NT + 4 * j) * ms + (j == NR - 1 ? vrl : vr));
    }
};

// acc(s) += C B for one AO set
template <int NT, int NR, int NS>
__device__ __forceinline__ void mma_set(MoAcc<NT, NR, NS>& acc, const COps<NT, NR>& c, int s, double b)
{
#pragma unroll
    for (int j = 0; j < NT; ++j) acc.t[j][s] = __builtin_amdgcn_mfma_f64_16x16x4f64(c.t[j], b, acc.t[j][s], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < NR; ++j) acc.r[j][s] = __builtin_amdgcn_mfma_f64_4x4x4f64(c.r[j], b, acc.r[j][s], 0, 0, 0);
}

// Rows R, R + 1, ... of the four standard shells: a K step each, its C operands
// in c, the next one's loaded before its MFMAs
template <int PASS, int L, bool SPH, int R, int NT, int NR, int NS>
__device__ __forceinline__ void quad_rows(const RowSets<L, SPH, PASS>& rows, const CWhere<NT, NR>& cw,
                                          const COps<NT, NR>& c, MoAcc<NT, NR, NS>& acc)
{
    if constexpr (R < shell_rows<L, SPH>()) {
        COps<NT, NR> next;
        if constexpr (R + 1 < shell_rows<L, SPH>()) cw.load(R + 1, next);
        double v[NS];
        rows.template row<R>(v);
#pragma unroll
        for (int s = 0; s < NS; ++s) mma_set(acc, c, s, v[s]);
        // a K step's values and operands are not hoisted above the one before
        // it: those of several rows at once do not fit beside the accumulators
        __builtin_amdgcn_sched_barrier(0);
        quad_rows<PASS, L, SPH, R + 1>(rows, cw, next, acc);
    }
}

// v = t on the lanes where on
template <int NS>
__device__ __forceinline__ void take(bool on, const double (&t)[NS], double (&v)[NS])
{
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = on ? t[s] : v[s];
}

// Rows of one (W = 4) or two (W = 2) standard shells left over at the end of
// their class, each held by W lane groups: group w of a shell's W (lane's w)
// gives row R + w to the K step, so the shell takes 1 / W of the K steps that a
// quad with empty places would.  `row`: the shell's first C row; c: row
// split_row(0, w).
template <int PASS, int W, int L, bool SPH, int R, int NT, int NR, int NS>
__device__ __forceinline__ void split_rows(const RowSets<L, SPH, PASS>& rows, CWhere<NT, NR>& cw, unsigned row, int w,
                                           const COps<NT, NR>& c, MoAcc<NT, NR, NS>& acc)
{
    constexpr int N = shell_rows<L, SPH>();
    if constexpr (R < N) {
        COps<NT, NR> next;
        if constexpr (R + W < N) {
            cw.shell(row + split_row<W>(R + W, w, N));
            cw.load(0, next);
        }
        double v[NS], t[NS];
        rows.template row<R>(v);
        auto place = [&](auto i) {
            constexpr int I = decltype(i)::value;
            if constexpr (I < W) {
                if constexpr (R + I < N) {
                    rows.template row<R + I>(t);
                } else {
#pragma unroll
                    for (int s = 0; s < NS; ++s) t[s] = 0.0;
                }
                take(w == I, t, v);
            }
        };
        place(std::integral_constant<int, 1>{});
        place(std::integral_constant<int, 2>{});
        place(std::integral_constant<int, 3>{});
#pragma unroll
        for (int s = 0; s < NS; ++s) mma_set(acc, c, s, v[s]);
        __builtin_amdgcn_sched_barrier(0);
        split_rows<PASS, W, L, SPH, R + W>(rows, cw, row, w, next, acc);
    }
}

// Rows of up to four shells with one general row map (T: nrow rows): set by set,
// the Cartesian values through the map.  The map comes through scalar loads, a
// row's C operands load while the row before it runs, and the fence keeps one
// set's values in registers at a time.  With each lane's own map read from memory
// and the accumulators in part in scratch 4 atoms x [s,s,p,d,f,g], 8 MOs, 48^3
// points took 41 us for rho, 109 with the gradient and 218 with the mixed second
// derivatives, now 32, 63 and 134.
template <int PASS, int L, int S, int NT, int NR, int NS>
__device__ __forceinline__ void quad_general(const OKMI_CONST double* T, int nrow, const ShellPows<L, double>& P, double S0,
                                             double S1, double S2, const CWhere<NT, NR>& cw, MoAcc<NT, NR, NS>& acc)
{
    if constexpr (S < NS) {
        constexpr int NC = ncart(L);
        double c[NC];
        cart_all<L, PassCodes<PASS>::c[S], double>(P, S0, S1, S2, c);
        COps<NT, NR> co, next;
        cw.load(0, co);
        for (int r = 0; r < nrow; ++r) {
            cw.load(min(r + 1, nrow - 1), next);
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < NC; ++k) v = fma(T[r * NC + k], c[k], v);
            mma_set(acc, co, S, v);
            co = next;
        }
        __builtin_amdgcn_sched_barrier(0);
        quad_general<PASS, L, S + 1>(T, nrow, P, S0, S1, S2, cw, acc);
    }
}

// Per-tile MO norms sum_p Phi_m(p)^2 over the tile's points (padding points
// excluded): column sums over the 16 lanes of each MO, the four columns
// added through LDS (red: 4 x MP doubles), one row of norm_part per tile.  Called by every thread.
template <int PASS, int U, bool STD>
__device__ __forceinline__ void tile_norms(const F64Args& a, int64_t tile, int col, int lane, bool act, double* red,
                                           const typename MoSplit<PASS, U, STD>::Acc& acc)
{
    using M = MoSplit<PASS, U, STD>;
    const int g = lane >> 4, n16 = lane & 15;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const double f = acc.get(u, 0);
        double v = act ? f * f : 0.0;
        v += __shfl_xor(v, 1);
        v += __shfl_xor(v, 2);
        v += __shfl_xor(v, 4);
        v += __shfl_xor(v, 8);
        if (n16 == 0) red[col * M::MP + 4 * u + g] = v;
    }
    __syncthreads();
    const int m = threadIdx.x;
    if (m < M::MP)
        a.norm_part[tile * M::MP + m] = (red[m] + red[M::MP + m]) + (red[2 * M::MP + m] + red[3 * M::MP + m]);
}

// Density terms of a pass at one point: sums over the MOs
template <int PASS> struct Terms {
    static constexpr int NS = PassCodes<PASS>::n;
    double r0 = 0.0;
    double t[NS > 1 ? NS - 1 : 1] = {};   // f0 f_s
    double u[6] = {};                     // f_x^2, f_y^2, f_z^2, f_x f_y, f_x f_z, f_y f_z
    static constexpr bool rho = PASS <= 1 || PASS == 4;
    static constexpr int NU = PASS == 1 ? 6 : PASS == 4 ? 3 : 0;

    template <typename F>
    __device__ __forceinline__ void each(bool second, F&& f)
    {
        if constexpr (rho) f(r0);
#pragma unroll
        for (int s = 0; s < NS - 1; ++s) f(t[s]);
        if (NU && second) {
#pragma unroll
            for (int q = 0; q < NU; ++q) f(u[q]);
        }
    }
};

// Density terms of the column from its MO values
template <int PASS, int U, bool STD>
__device__ __forceinline__ void epilogue_f64(const F64Args& a, const TileWhere& W, const double* occ, int col, int lane,
                                             const typename MoSplit<PASS, U, STD>::Acc& acc)
{
    constexpr int NS = PassCodes<PASS>::n;
    const int g = lane >> 4, n16 = lane & 15;
    const bool second = PASS == 4 || (PASS == 1 && a.need_mask >> 4);   // uniform: f_a f_b halves wanted
    Terms<PASS> T;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        // padding MOs repeat the last one's values and weigh nothing
        const double w = occ[4 * u + g];
        double f[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) f[s] = acc.get(u, s);
        const double wf = w * f[0], w2f = 2.0 * wf;
        if constexpr (Terms<PASS>::rho) T.r0 = fma(wf, f[0], T.r0);
#pragma unroll
        for (int s = 1; s < NS; ++s) T.t[s - 1] = fma(w2f, f[s], T.t[s - 1]);
        if constexpr (PASS == 1 || PASS == 4) {
            if (second) {
                const double wx = 2.0 * w * f[1], wy = 2.0 * w * f[2], wz = 2.0 * w * f[3];
                T.u[0] = fma(wx, f[1], T.u[0]);
                T.u[1] = fma(wy, f[2], T.u[1]);
                T.u[2] = fma(wz, f[3], T.u[2]);
                if constexpr (PASS == 1) {
                    T.u[3] = fma(wx, f[2], T.u[3]);
                    T.u[4] = fma(wx, f[3], T.u[4]);
                    T.u[5] = fma(wy, f[3], T.u[5]);
                }
            }
        }
    }
    T.each(second, [](double& v) {
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
    });
    int64_t p;
    const bool act = W.index(a, col * 16 + n16, p);
    if (g == 0 && act) {
        // (a launch over further MOs adds to what the one before it wrote)
        auto out = [&](double* o, double v) { *o = a.add ? *o + v : v; };
        if constexpr (Terms<PASS>::rho) out(a.rho + p, T.r0);
#pragma unroll
        for (int s = 1; s < NS; ++s) {
            const int code = PassCodes<PASS>::c[s];
            double v = T.t[s - 1];
            if (PASS == 4 && s > 3) v += T.u[s - 4];   // f0 f_aa + f_a^2
            if (a.need_mask >> code & 1) out(a.term + a.term_row[code] * a.ld_term + p, v);
        }
        if constexpr (PASS == 1) {
#pragma unroll
            for (int q = 0; q < 6; ++q)
                if (a.need_mask >> (4 + q) & 1) out(a.term2 + (4 + q) * a.ld_term + p, T.u[q]);
        }
    }
}

// MO values of the column, [row of the code][mo][point]
template <int PASS, int U, bool STD>
__device__ __forceinline__ void store_mos(const F64Args& a, const TileWhere& W, int col, int lane,
                                          const typename MoSplit<PASS, U, STD>::Acc& acc)
{
    const int g = lane >> 4, n16 = lane & 15;
    int64_t p;
    if (!W.index(a, col * 16 + n16, p)) return;
#pragma unroll
    for (int s = 0; s < PassCodes<PASS>::n; ++s) {
        const int code = PassCodes<PASS>::c[s];
        if (!(a.need_mask >> code & 1)) continue;   // uniform
        double* out = a.term + a.term_row[code] * a.ld_set + p;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int m = 4 * u + g;
            if (m < a.nmo) out[m * a.ld_term] = acc.get(u, s);
        }
    }
}

// The list's entries from s on that are of class L, KIND, at the wave's points
// (lane: px, py, pz), evaluated and contracted: with W = 1 four at a time (three
// at the end; general row maps: those with the map of the first), with W = 2 the
// two and with W = 4 the one left over.  One loop per case, in the list's order:
// with the cases as branches of a single loop the compiler moved the accumulators
// through scratch.
template <int PASS, int U, bool STD, int L, int KIND, int W>
__device__ __forceinline__ void class_loop(const F64Args& a, const LiveShell* ent, int& s, int cnt, int base, double px,
                                           double py, double pz, int g, CWhere<U / 4, U % 4>& cw,
                                           typename MoSplit<PASS, U, STD>::Acc& acc)
{
    using M = MoSplit<PASS, U, STD>;
    constexpr bool need1 = PASS == 1 || PASS == 2 || PASS == 4, need2 = PASS >= 2;
    // leftovers have cases of their own (not where the rows take most registers)
    constexpr bool split = L > 0 && KIND != SHELL_T_GENERAL && PASS != 3;
    if constexpr (W == 1 || split) while (s < cnt) {
        int at = min(s + g, cnt - 1);   // lane's entry
        const unsigned idcls = ent[at].idcls, cls = __builtin_amdgcn_readfirstlane(idcls >> LIST_ID_BITS);
        const unsigned kind = cls >> 3 & 3;
        if ((cls & 7) != L || kind != KIND) return;
        bool mine = s + g < cnt && idcls >> LIST_ID_BITS == cls;
        int t0 = 0;   // general row maps: shells with the same one
        if constexpr (KIND == SHELL_T_GENERAL) {
            t0 = __builtin_amdgcn_readfirstlane(ent[at].t0);
            mine = mine && ent[at].t0 == t0;
        }
        const int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(mine)) >> 4;
        if (W == 1 ? split && n < 3 : n != 4 / W) return;
        const int w = g & (W - 1);
        // lanes without a shell repeat the first one with no primitive
        if (W > 1) at = s + g / W;
        else if (!mine) at = s;
        const LiveShell* e = ent + at;
        const unsigned rowlive = e->rowlive;
        const int live = W > 1 || mine ? rowlive >> LIST_ROW_BITS : 0;
        s += n;
        const unsigned row = rowlive & LIST_ROW_MASK;
        if constexpr (W > 1) cw.shell(row + split_row<W>(0, w, shell_rows<L, KIND == SHELL_T_SPHERICAL>()));
        else cw.shell(row);
        COps<M::NT, M::NR> c;
        cw.load(0, c);
        const double X = px - e->c[0], Y = py - e->c[1], Z = pz - e->c[2];
        const double rr = X * X + Y * Y + Z * Z;
        double S0 = 0.0, S1 = 0.0, S2 = 0.0;
        auto prim = [&](double alpha, double d) {
            const double de = d * gauss_f64(alpha * rr);
            S0 += de;
            if constexpr (need1) S1 = fma(alpha, de, S1);
            if constexpr (need2) S2 = fma(alpha * alpha, de, S2);
        };
        // as many primitives as one of the four has in reach (their radii descend)
#pragma nounroll
        for (int q = 0; q < 4; ++q) {
            if (__builtin_amdgcn_ballot_w64(live > q) == 0) break;
            const double alpha = e->alpha[q], d = e->d[q];
            prim(alpha, live > q ? d : 0.0);
        }
        if (__builtin_amdgcn_ballot_w64(live == 4) != 0) {   // all four in reach: those past them
            const ListRec* sh = a.shells + base + (e->idcls & LIST_ID_MASK);
#pragma nounroll
            for (int q = 4;; ++q) {
                const PrimGroup* pg = a.more + sh->more + ((q - 4) >> 2);
                const bool on = live == 4 && q < sh->nprim && e->d2 < pg->rcut2[q & 3];
                if (__builtin_amdgcn_ballot_w64(on) == 0) break;
                prim(on ? pg->alpha[q & 3] : 0.0, on ? pg->d[q & 3] : 0.0);
            }
        }
        S1 *= -2.0;
        S2 *= 4.0;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (KIND == SHELL_T_GENERAL) {
            ShellPows<L, double> P;
            P.init(X, Y, Z);
            quad_general<PASS, L, 0>(cptr(a.T) + t0, (int)(cls >> 5), P, S0, S1, S2, cw, acc);
        } else {
            const RowSets<L, KIND == SHELL_T_SPHERICAL, PASS> rows(X, Y, Z, S0, S1, S2);
            constexpr bool SPH = KIND == SHELL_T_SPHERICAL;
            if constexpr (W > 1) split_rows<PASS, W, L, SPH, 0>(rows, cw, row, w, c, acc);
            else quad_rows<PASS, L, SPH, 0>(rows, cw, c, acc);
        }
    }
}

// STD: for bases of standard shells (l <= 3, real spherical or Cartesian rows)
template <int PASS, int U, bool STD, bool MO>
__global__ __launch_bounds__(256, (MoSplit<PASS, U, STD>::OCC)) void k_fused_f64(F64Args a)
{
    using M = MoSplit<PASS, U, STD>;
    constexpr int MP = M::MP, LCAP = M::LCAP, NW = M::NW;
    __shared__ LiveShell ent[LCAP];      // shells in reach of the tile
    __shared__ double occ[MP];           // occupations, zero padded
    __shared__ double sbox[6];
    __shared__ double norms[MO ? 1 : NW * MP];
    __shared__ int wsum[NW];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, n16 = lane & 15;
    const unsigned tile = a.tile0 + blockIdx.x;
    const TileWhere W(a, tile);
    double px, py, pz;
    W.point(a, lane, px, py, pz);   // lane l of every wave: point l of the tile, for its box
    double qx, qy, qz;
    W.point(a, 16 * wave + n16, qx, qy, qz);   // the wave's 16 points
    shared_box(wave, px, py, pz, sbox);
    if (!MO && threadIdx.x < MP) occ[threadIdx.x] = (int)threadIdx.x < a.nmo ? a.occ[threadIdx.x] : 0.0;
    __syncthreads();

    typename M::Acc acc;
    acc.zero();
    CWhere<M::NT, M::NR> cw(a, MP, n16);
    int t0 = 0;
    while (t0 < a.nsh) {
        // shells in reach, as many as the list holds
        const int base = t0;
        int cnt = 0;
        while (t0 < a.nsh && t0 - base < (int)LIST_ID_MASK - LCAP) {
            const int n = append_live<LCAP, NW>(a.shells, a.nsh, t0, base, sbox, ent, wsum, cnt);
            __syncthreads();
            if (n < 0) break;
            cnt += n;
            t0 += LCAP;
        }
        int s = 0;
#define OKMI_LOOP(L, KIND, W) class_loop<PASS, U, STD, L, KIND, W>(a, ent, s, cnt, base, qx, qy, qz, g, cw, acc)
#define OKMI_CLASS(L, KIND)        \
    OKMI_LOOP(L, KIND, 1);         \
    OKMI_LOOP(L, KIND, 2);         \
    OKMI_LOOP(L, KIND, 4)
        if constexpr (!STD) {
            OKMI_CLASS(4, SHELL_T_CARTESIAN);
            OKMI_LOOP(4, SHELL_T_GENERAL, 1);
        }
        OKMI_CLASS(3, SHELL_T_CARTESIAN);
        OKMI_CLASS(3, SHELL_T_SPHERICAL);
        if constexpr (!STD) OKMI_LOOP(3, SHELL_T_GENERAL, 1);
        OKMI_CLASS(2, SHELL_T_CARTESIAN);
        OKMI_CLASS(2, SHELL_T_SPHERICAL);
        if constexpr (!STD) OKMI_LOOP(2, SHELL_T_GENERAL, 1);
        OKMI_CLASS(1, SHELL_T_CARTESIAN);
        if constexpr (!STD) OKMI_LOOP(1, SHELL_T_GENERAL, 1);
        OKMI_LOOP(0, SHELL_T_CARTESIAN, 1);
        if constexpr (!STD) OKMI_LOOP(0, SHELL_T_GENERAL, 1);
#undef OKMI_CLASS
#undef OKMI_LOOP
        if (t0 < a.nsh) __syncthreads();   // (uniform) the list is read before it is filled again
    }
    if constexpr (MO) {
        store_mos<PASS, U, STD>(a, W, wave, lane, acc);
    } else {
        epilogue_f64<PASS, U, STD>(a, W, occ, wave, lane, acc);
        if constexpr (PASS <= 1 || PASS == 4) {
            if (a.norm_part) {   // uniform: every thread takes the branch or none
                int64_t p;
                const bool act = W.index(a, wave * 16 + n16, p);
                tile_norms<PASS, U, STD>(a, tile, wave, lane, act, norms, acc);
            }
        }
    }
}

template <int PASS, bool STD, int U, bool MO>
int launch_f64_one(F64Args a, hipStream_t st)
{
    if (a.ntile >= ((int64_t)1 << 31)) {   // one workgroup per tile; brick indices are 32-bit
        okmi_set_error("rho_fused: %lld tiles of 64 points (at most 2^31 - 1 per call)", (long long)a.ntile);
        return 1;
    }
    OkmiProfScope prof(MO ? "mo_fused_f64" : "rho_fused_f64", st);
    // (a launch holds fewer than 2^32 threads)
    for (int64_t t = 0; t < a.ntile; t += OKMI_MAX_BLOCKS) {
        a.tile0 = (unsigned)t;
        const unsigned n = (unsigned)std::min(a.ntile - t, OKMI_MAX_BLOCKS);
        hipLaunchKernelGGL((k_fused_f64<PASS, U, STD, MO>), dim3(n), dim3(256), 0, st, a);
    }
    return 0;
}

// One launch with the smallest of the instances U... (ascending) that holds
// a.units groups of 4 MOs
template <int PASS, bool STD, bool MO, int U, int... MORE>
int launch_f64_units(const F64Args& a, hipStream_t st)
{
    if (a.units <= U) return launch_f64_one<PASS, STD, U, MO>(a, st);
    if constexpr (sizeof...(MORE) > 0) {
        return launch_f64_units<PASS, STD, MO, MORE...>(a, st);
    } else {
        okmi_set_error("rho_fused: no instance for %d groups of 4 MOs", a.units);
        return 1;
    }
}

}  // namespace okmi_fused
