// FP64 fused density and MO values (fused_f64.h): the launch sequences.
#include "fused_tile.h"

namespace okmi_fused {
namespace {

// mo_norm[m] += sum over tiles of part[tile][m], m < nmo: one workgroup per
// MO, each thread a fixed stride of tiles, then a tree in LDS (the order of
// the additions does not depend on timing)
__global__ void k_norm_reduce(const double* part, int64_t ntile, int mpad, int nmo, double* mo_norm)
{
    __shared__ double red[256];
    const int m = blockIdx.x;
    double s = 0.0;
    for (int64_t t = threadIdx.x; t < ntile; t += 256) s += part[t * mpad + m];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0 && m < nmo) mo_norm[m] += red[0];
}

}  // namespace

int launch_norm_reduce(const double* part, int64_t ntile, int mpad, int nmo, double* mo_norm, hipStream_t st)
{
    if (ntile <= 0 || nmo <= 0) return 0;
    hipLaunchKernelGGL(k_norm_reduce, dim3((unsigned)nmo), dim3(256), 0, st, part, ntile, mpad, nmo, mo_norm);
    return 0;
}

int launch_rho_f64(F64Args a, int u, int pass, bool standard, hipStream_t st)
{
    a.units = f64_units(u, pass, standard, false);
    if (!standard) return launch_f64_general(a, pass, st);
    switch (pass) {
    case 0: return launch_f64_p0(a, st);
    case 1: return launch_f64_p1(a, st);
    case 4: return launch_f64_p4(a, st);
    default: return launch_f64_p23(a, pass, st);
    }
}

}  // namespace okmi_fused

namespace {

using namespace okmi_fused;

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// C [nmo][nao] -> [group][nao][width], group g its MOs from `step` g on, zero
// padded: one 32 x 32 block per workgroup of 256 threads, through LDS.  (A matrix
// per group: rows of at most 64 MOs, which the kernel's 32-bit offsets reach for
// any basis; rows of all MOs passed 4 GiB at 25,000 AOs x 21,500 MOs.)
__global__ __launch_bounds__(256) void k_transpose_c(const double* C, int nmo, int nao, int step, int width, double* out)
{
    __shared__ double t[32][33];
    const int r0 = 32 * blockIdx.x, m0 = 32 * blockIdx.y, g0 = step * blockIdx.z;
    const int have = min(step, nmo - g0);
    C += (int64_t)g0 * nao;
    out += (int64_t)blockIdx.z * nao * width;
    for (int i = threadIdx.x; i < 1024; i += 256) {
        const int m = m0 + i / 32, r = r0 + i % 32;
        t[i / 32][i % 32] = m < have && r < nao ? C[(int64_t)m * nao + r] : 0.0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 1024; i += 256) {
        const int r = r0 + i / 32, m = m0 + i % 32;
        if (r < nao && m < width) out[(int64_t)r * width + m] = t[i % 32][i / 32];
    }
}

// Whether C is transposed first, for `tiles` tiles over all passes and u groups of
// 4 MOs.  The transposition and its launch take about 3 us.  From 512 tiles on
// reading the caller's C costs more: a tile about 8 ns over whole lines of C^T.
// Rho alone has little work between the loads of its K steps, 64 lines per 16 MOs
// where C^T has 8, the more so where a row of C is whole lines of 128 bytes, which
// share the sets of the vector cache: with more tiles than CUs it pays from 17
// MOs and 160 AOs on (20 atoms, 400 AOs, 40 MOs, 20,000 points: 94 us in place, 50
// from C^T; rows of other lengths from about 360 AOs on), with fewer where two or
// three groups of 4 MOs add loads of their own (400 AOs, 8,192 points, 28 MOs: 52
// and 44; 56 MOs: 62 and 44; 32 MOs: 36 and 40; 440 AOs, 60 MOs: 60 and 50).
bool transposed(int64_t tiles, int u, int nao, bool rho_alone)
{
    if (tiles >= 512) return true;
    const bool lines = nao % 16 == 0;
    if (!rho_alone || u < 5 || nao < (lines ? 160 : 360)) return false;
    if (tiles > 256) return true;
    return lines ? u >= 7 && u % 4 >= 2 : u >= 11 && u % 4 == 3;
}

// Per point: up to 20 term rows; with MO norms one row of per-tile norms per
// 64 points (at most 64 MOs a launch)
constexpr size_t PT_BYTES = 20 * 8, NORM_PT_BYTES = 8;

// The passes of a request, and its MOs in equal groups of at most as many as a
// pass holds in registers: 64 at up to four AO sets, 40 at seven.
struct Plan {
    bool standard, p1, p2, p3, p4;
    bool direct;            // every output a first or diagonal second derivative, each once
    int need, groups, u;    // codes; launches over 4 u MOs each

    Plan(const OkmiBasis* b, int nmo, const int* drv_out, int nout) : standard(b->standard), direct(true), need(0)
    {
        for (int r = 0; r < nout; ++r) {
            const int d = drv_out[r];
            if (d < 1 || d > 6 || (need >> d & 1)) direct = false;
            need |= 1 << d;
        }
        p1 = (need & ~1) != 0;
        p2 = (need & (7 << 4)) != 0;
        p3 = (need & (7 << 7)) != 0;
        // diagonal second derivatives and no mixed ones: all seven AO sets at
        // once (bases with general row maps up to the MOs of one launch)
        p4 = p2 && !p3 && (standard || nmo <= 40);
        if (p2 && !p4) direct = false;
        const int cap = p4 ? 40 : 64;
        groups = (nmo + cap - 1) / cap;
        u = ((nmo + groups - 1) / groups + 3) / 4;
    }
    int first() const { return p4 ? 4 : p1 ? 1 : 0; }
    // MOs of a launch of a pass, and of a group's C^T (the padding of every pass)
    int64_t mp(int pass) const { return 4 * (int64_t)f64_units(u, pass, standard, false); }
    int64_t width() const { return std::max(mp(first()), (p2 && !p4) || p3 ? mp(3) : 0); }
    size_t c_bytes(const OkmiBasis* b, int nmo) const
    {
        const size_t n = align256(8 * (size_t)b->nao * groups * width());
        return nmo <= 64 ? std::max(n, okmi_fused_c_bytes(b, nmo, OKMI_PREC_F64)) : n;
    }
    size_t slack(bool norms) const { return 256 + (norms ? 256 + (size_t)mp(first()) * 8 : 0); }
};

F64Args basis_args(const OkmiBasis* b, const GridDesc& g, int nmo, const double* d_c)
{
    F64Args f{};
    f.shells = b->d_lshells;
    f.more = b->d_lgroups;
    f.nsh = b->nshell;
    f.T = b->d_T;
    f.grid = g;
    f.nmo = nmo;
    f.nao = b->nao;
    f.C = d_c;
    for (int c = 0; c < 10; ++c) f.term_row[c] = c;
    return f;
}

void transpose_c(const OkmiBasis* b, const double* d_c, int nmo, int groups, int step, int64_t width, double* out,
                 hipStream_t st)
{
    hipLaunchKernelGGL(k_transpose_c, dim3((unsigned)((b->nao + 31) / 32), (unsigned)((width + 31) / 32), (unsigned)groups),
                       dim3(256), 0, st, d_c, nmo, b->nao, step, (int)width, out);
}

}  // namespace

// More than 64 MOs: the groups follow one another in the fused kernel and share
// a launch in the staged one, so a few tiles leave the fused one's launches short
// of work, the more groups there are the longer.  Fused / staged time over 20 to
// 200 atoms at 1 to 64 and at 216 tiles: rho, with and without first derivatives,
// 2 groups 0.5 to 1.2 and 0.3 to 0.6, 4 groups 0.9 to 2.4 and 0.5 to 0.8, 32 groups
// 1.0 to 4.2 and 0.7; diagonal second derivatives, 5 groups 0.6 to 1.1 and 0.2 to
// 0.5, 20 groups 1.1 to 2.2 and 0.4 to 0.7; mixed ones up to 1.3 and up to 0.4.
bool okmi_rho_f64_fused_pays(const OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, int nmo, const int* drv_out,
                             int nout)
{
    const Plan pl(b, nmo, drv_out, nout);
    F64Args f{};
    f.grid = g;
    f.np = np;
    f.set_bricks(g.regular && p0 == 0 && np == g.nx * g.ny * g.nz);
    return f.ntile >= 128 || pl.p3 || pl.groups < (pl.p4 ? 10 : 4);
}

size_t okmi_rho_f64_fused_min_bytes(const OkmiBasis* b, int nmo, const int* drv_out, int nout, bool norms)
{
    const Plan pl(b, nmo, drv_out, nout);
    return pl.c_bytes(b, nmo) + pl.slack(norms) + (PT_BYTES + (norms ? NORM_PT_BYTES : 0)) * 64;
}

int okmi_launch_rho_f64_fused(const OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, const double* d_c,
                              const double* d_occ, int nmo, const int* drv_out, int nout, double* rho, double* delta,
                              int64_t ld_delta, double* mo_norm, void* ws, size_t ws_bytes, hipStream_t st)
{
    for (int r = 0; r < nout; ++r)
        if (drv_out[r] < 0 || drv_out[r] > 9) {
            okmi_set_error("The selection `drv=%d` is not valid!", drv_out[r]);
            return 1;
        }
    const Plan pl(b, nmo, drv_out, nout);
    const int64_t mp = pl.mp(pl.first()), step = 4 * (int64_t)pl.u;   // MO norms of a tile; MOs of a group
    const size_t fixed = pl.c_bytes(b, nmo), least = okmi_rho_f64_fused_min_bytes(b, nmo, drv_out, nout, mo_norm != nullptr);
    if (!ws || ws_bytes < least) {
        okmi_set_error("rho_fused: workspace of %zu bytes is too small (need at least %zu)", ws_bytes, least);
        return 1;
    }
    // per point: the term rows, plus the per-tile MO norms (mp doubles per
    // 64-point tile) when wanted
    const size_t per_pt = PT_BYTES + (mo_norm ? NORM_PT_BYTES : 0);
    const size_t avail = ws_bytes - fixed - pl.slack(mo_norm != nullptr);
    // a whole regular grid whose buffers fit is tiled in 4x4x4 bricks (the
    // faces may add tiles beyond np / 64); outputs written where they belong
    // need no term rows
    const size_t term_bytes = pl.direct ? 0 : PT_BYTES;
    const int64_t nbrick = ((g.nx + 3) / 4) * ((g.ny + 3) / 4) * ((g.nz + 3) / 4);
    const bool brick = g.regular && p0 == 0 && np == g.nx * g.ny * g.nz &&
                       term_bytes * (size_t)np + (mo_norm ? (size_t)nbrick * mp * 8 : 0) <= avail;
    int64_t chunk = brick ? np : std::min<int64_t>(np, (int64_t)(avail / per_pt) & ~(int64_t)63);
    if (chunk <= 0) chunk = np;   // unreachable: avail holds 64 points
    char* w = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
    double* ct = (double*)w;
    double* term = (double*)(w + fixed);
    double* norm_part = mo_norm ? (double*)(w + fixed + align256(term_bytes * (size_t)chunk)) : nullptr;

    F64Args f = basis_args(b, g, nmo, d_c);
    f.need_mask = pl.need;
    f.np = std::min(np, chunk);
    f.set_bricks(brick);
    if (pl.groups > 1 || transposed(f.ntile * (1 + (pl.p2 && !pl.p4) + pl.p3), pl.u, b->nao, pl.first() == 0)) {
        transpose_c(b, d_c, nmo, pl.groups, (int)step, pl.width(), ct, st);
        f.ct_ld = (int)pl.width();
    }
    if (pl.direct) {
        f.ld_term = ld_delta;
        for (int r = 0; r < nout; ++r) f.term_row[drv_out[r]] = r;
    } else {
        f.term = term;
        f.term2 = term + 10 * chunk;
        f.ld_term = chunk;
    }
    for (int64_t c0 = 0; c0 < np; c0 += chunk) {
        const int64_t n = std::min(np - c0, chunk);
        f.p0 = p0 + c0;
        f.np = n;
        if (!brick) f.set_bricks(false);
        f.rho = rho + c0;
        if (pl.direct) f.term = delta + c0;
        for (int gr = 0; gr < pl.groups; ++gr) {
            const int m0 = gr * (int)step;
            if (m0 >= nmo) break;
            f.add = gr > 0;
            f.nmo = std::min<int>(nmo - m0, (int)step);
            f.C = d_c + (int64_t)m0 * b->nao;
            f.occ = d_occ + m0;
            if (f.ct_ld) f.ct = ct + (int64_t)gr * b->nao * f.ct_ld;
            f.norm_part = norm_part;   // read by the first pass (rho) only
            int r = launch_rho_f64(f, pl.u, pl.first(), b->standard, st);
            if (!r && pl.p2 && !pl.p4) r = launch_rho_f64(f, pl.u, 2, b->standard, st);
            if (!r && pl.p3) r = launch_rho_f64(f, pl.u, 3, b->standard, st);
            if (!r && mo_norm) r = launch_norm_reduce(norm_part, f.ntile, (int)mp, f.nmo, mo_norm + m0, st);
            if (r) return r;
        }
        if (!pl.direct)
            okmi_launch_gather(rho + c0, term, pl.p4 ? nullptr : f.term2, chunk, drv_out, nout, delta + c0, ld_delta, n, st);
    }
    return okmi_check_launch("rho_fused");
}

size_t okmi_mo_f64_fused_bytes(const OkmiBasis* b, int nmo)
{
    return 256 + align256(8 * (size_t)b->nao * ((nmo + 63) / 64 * 64 + 4));
}

// Codes in passes {0,x,y,z}, {0,xx,yy,zz}, {0,xy,xz,yz} (code 0 alone: {0}), MOs
// in equal groups of at most 64.  Screened with the bound of the AO kernel
// (OKMI_SCREEN), as MO values are wanted far from the molecule too.
int okmi_launch_mo_f64_fused(const OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, const int* drv, int ndrv,
                             const double* d_c, int nmo, double* d_mo, int64_t ld_mo, void* ws, hipStream_t st)
{
    const int groups = (nmo + 63) / 64, u = ((nmo + groups - 1) / groups + 3) / 4, step = 4 * u;
    double* ct = (double*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
    const int64_t width = 4 * (int64_t)f64_units(u, 3, b->standard, true);   // (the widest instance's)
    transpose_c(b, d_c, nmo, groups, step, width, ct, st);
    F64Args f = basis_args(b, g, nmo, d_c);
    f.shells = b->d_lshells_a;
    f.more = b->d_lgroups_a;
    f.ct_ld = (int)width;
    f.p0 = p0;
    f.np = np;
    f.set_bricks(g.regular && p0 == 0 && np == g.nx * g.ny * g.nz);
    f.ld_term = ld_mo;
    f.ld_set = (int64_t)nmo * ld_mo;
    int left = 0;
    for (int j = 0; j < ndrv; ++j) {
        left |= 1 << drv[j];
        f.term_row[drv[j]] = j;
    }
    for (int pass = 0; pass <= 3; ++pass) {
        static constexpr int codes[4] = {1, 0xf, 0x71, 0x381};
        // code 0 by the first pass that takes a derivative, or alone
        if (pass == 0 ? left != 1 : (left & codes[pass] & ~1) == 0) continue;
        f.need_mask = left & codes[pass];
        left &= ~codes[pass];
        for (int gr = 0; gr < groups; ++gr) {
            const int m0 = gr * step;
            if (m0 >= nmo) break;
            f.nmo = std::min(nmo - m0, step);
            f.ct = ct + (int64_t)gr * b->nao * width;
            f.term = d_mo + (int64_t)m0 * ld_mo;
            f.units = f64_units(u, pass, b->standard, true);
            const int r = launch_mo_f64(f, pass, b->standard, st);
            if (r) return r;
        }
    }
    return okmi_check_launch("mo_eval");
}
