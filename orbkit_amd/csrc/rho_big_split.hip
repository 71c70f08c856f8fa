// Density for many MOs at the split-bf16 precisions, rho and rho with first
// derivatives (S = 1 and 4 AO sets; rho_big.hip has the other requests).
// Replaces slice_rho's density branch (orbkit/core.py:179-308).  Per chunk of
// points:
//   1. k_live_quads lists, per tile of NP points, the 32-row chunks of the fused
//      row order with a shell in reach, and which of their quads (four
//      consecutive rows) hold a row of such a shell;
//   2. k_ao_live writes the AO sets in FP32 in tiles of 64 points,
//      ao[tile of 64][set][row][64], rows of dead quads left unwritten;
//   3. k_rho_split contracts the listed chunks with C, one K step of the bf16
//      MFMA each, and reduces its MOs to density terms;
//   4. k_reduce_big sums the MO blocks in a fixed order.
//
// Bound by a K step's phases: the matrix cores are busy 43% of the launch, LDS
// 22%, the other VALU work 18%, and the two workgroups of a CU overlap them in
// part.  Before, one workgroup of 128 MOs filled a CU (129 KB of LDS), each of
// the two waves on a column split the AO tile again, and the fourth MO block of
// 400 MOs staged and split everything for its 16 MOs.  Now a workgroup of four
// waves splits the tile once, on its way to LDS, and holds up to 80 MOs (five
// tiles of 16 per wave, spread evenly: 400 MOs are five full blocks), so that
// two workgroups share a CU (64 KB each); a chunk's dead quads are not loaded,
// and the AO rows of a tile lie together.  200 atoms, 2,950 AOs, 400 MOs, 128^3
// points: 22.9 -> 14.9 ms (eight waves of 64 MOs x 16 points in one workgroup
// per CU, two LDS stages: 16.0).  Chunks stay whole K steps: eight live quads
// of several chunks to a K step took 8.8 ms with the same error, but another
// order of the FP32 sums.
#include "rho_big.h"

namespace {

using namespace okmi_split;

constexpr int QR = 4;     // rows per quad
constexpr int KS = 32;    // rows per chunk, one K step

template <int PREC, int S, int T>
struct SplitCfg {
    static constexpr int NPL = PREC == OKMI_PREC_BF16X6 ? 3 : 2;
    static constexpr int NP = S == 1 ? 128 : 64;       // points per workgroup
    static constexpr int NPW = NP / 64;                // 16-point columns per wave
    static constexpr int U = S * NP / 64;              // 8-row x 64-point units a wave stages per K step
    static constexpr int MB = 16 * T;                  // MOs per workgroup
    static constexpr int CPW = NPL * MB;               // 16-byte pieces of C a wave stages per K step
    static constexpr int CR = (CPW + 63) / 64;
    // 16-byte slots: AO [S][NPL][4][NP], C [4][NPL][MB]; reads and writes of 16
    // lanes fall in 256 consecutive bytes
    static constexpr int AO_SLOTS = S * NPL * 4 * NP, C_SLOTS = 4 * NPL * MB;
};

struct SplitArgs {
    const float* ao;         // [tile of 64][S][kpad][64]
    int64_t kpad;
    int64_t sub;             // tiles of 64 in ao
    int64_t np;              // points in this chunk
    const void* C;           // [octet of rows][plane][mpad][8] bf16
    int64_t mpad;            // MOs in whole tiles of 16
    const double* occ;       // [mpad], zero padded
    double* partial;         // [nb][S][ld]
    int64_t ld;
    int nb, nt;              // MO blocks, MO tiles of 16
    const int* list;         // [tile][kpad / 32] live chunks: chunk << 8 | its live quads
    const int* count;        // [tile]
    int64_t nblocks;
};

// K loop over the live chunks of point tile tn for the NV MO tiles from MO m0 on
template <int PREC, int S, int T, int NV>
__device__ __forceinline__ void split_loop(const SplitArgs& a, bf8* smem, int64_t tn, int m0, int steps, int lane, int wave,
                                           f4 (&acc)[T][SplitCfg<PREC, S, T>::NPW][S])
{
    using P = SplitCfg<PREC, S, T>;
    constexpr int NPL = P::NPL, NP = P::NP, NPW = P::NPW, U = P::U, MB = P::MB;
    const int g = lane >> 4, n16 = lane & 15;
    // ---- staging: wave w takes rows 8 w .. 8 w + 7 of a chunk (two quads):
    // their C and U units of 8 rows x 64 points
    const int* list = a.list + tn * (a.kpad / KS);
    auto entries = [&](int w) { return list[min(64 * w + lane, steps - 1)]; };
    // two windows of 64 entries across the lanes
    int lv0 = entries(0), lv1 = entries(1), win = 0;
    // unit u: set u of 4, or 64-point tile u of 2 (the last one again past the end)
    const int64_t sub = S == 1 ? min((int64_t)1, a.sub - 1 - 2 * tn) * a.kpad * 64 : a.kpad * 64;
    const float* ao = a.ao + tn * (NP / 64) * (S * a.kpad * 64) + lane;
    int coff[P::CR];   // elements from an octet's planes
#pragma unroll
    for (int r = 0; r < P::CR; ++r) {
        const int e = min(64 * r + lane, P::CPW - 1);
        coff[r] = (int)((e / MB) * a.mpad + min((int64_t)(m0 + e % MB), a.mpad - 1)) * 8;
    }
    float x[U][8];
    bf8 cp[P::CR];
    unsigned live = 0;   // the live ones of the two quads being loaded
    auto load = [&](int st) {
        if (st >> 6 != win) {   // (chunks are taken in order)
            win = st >> 6;
            lv0 = lv1;
            lv1 = entries(win + 1);
        }
        const unsigned e = __builtin_amdgcn_readlane(lv0, st & 63);
        const int k0 = 4 * (int)(e >> 8) + wave;
        live = (e >> 2 * wave) & 3;
        // dead quads are not read: a live one of the chunk in their place
        const int any = KS * (int)(e >> 8) + QR * __builtin_ctz(e & 0xff);
        const int r0 = live & 1 ? 8 * k0 : any, r1 = live & 2 ? 8 * k0 + QR : any;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j) x[u][j] = ao[u * sub + ((j < 4 ? r0 : r1) + (j & 3)) * 64];
        const __bf16* c0 = (const __bf16*)a.C + (int64_t)k0 * (NPL * 8) * a.mpad;
#pragma unroll
        for (int r = 0; r < P::CR; ++r) cp[r] = *(const bf8*)(c0 + coff[r]);
    };
    auto put = [&] {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = live & (j < 4 ? 1 : 2) ? x[u][j] : 0.f;   // (dead quads: zero rows)
            Split<PREC> sp;
            split8<PREC>(v, sp);
            const int s = S == 1 ? 0 : u, half = S == 1 ? u : 0;
#pragma unroll
            for (int pl = 0; pl < NPL; ++pl) smem[((s * NPL + pl) * 4 + wave) * NP + 64 * half + lane] = sp.p[pl];
        }
        bf8* d = smem + P::AO_SLOTS + wave * P::CPW;
#pragma unroll
        for (int r = 0; r < P::CR; ++r)
            if (64 * r + 63 < P::CPW || 64 * r + lane < P::CPW) d[64 * r + lane] = cp[r];
    };
    load(0);
    for (int st = 0; st < steps; ++st) {
        if (st > 0) __syncthreads();   // the chunk before is read
        put();
        load(min(st + 1, steps - 1));
        __syncthreads();
        const bf8* as = smem + P::AO_SLOTS + g * P::CPW + n16;
        Split<PREC> A[NV], B[2];
        auto read_b = [&](int i, Split<PREC>& o) {   // operand i = column * S + set
            const int c = i / S, s = i % S;
#pragma unroll
            for (int pl = 0; pl < NPL; ++pl) o.p[pl] = smem[((s * NPL + pl) * 4 + g) * NP + (wave * NPW + c) * 16 + n16];
        };
        read_b(0, B[0]);
#pragma unroll
        for (int rb = 0; rb < NV; ++rb)
#pragma unroll
            for (int pl = 0; pl < NPL; ++pl) A[rb].p[pl] = as[pl * MB + 16 * rb];
#pragma unroll
        for (int i = 0; i < NPW * S; ++i) {
            if (i + 1 < NPW * S) read_b(i + 1, B[(i + 1) & 1]);
            const Split<PREC>& b = B[i & 1];
            const int c = i / S, s = i % S;
            // term by term over the MO tiles, in mfma_split's order: two
            // products of one accumulator are NV apart
            constexpr int NT = NPL == 3 ? 6 : 3;
            constexpr int ta[6] = {NPL == 3 ? 2 : 1, NPL == 3 ? 1 : 0, 0, 1, 0, 0};
            constexpr int tb[6] = {0, 1, NPL == 3 ? 2 : 0, 0, 1, 0};
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int rb = 0; rb < NV; ++rb)
                    acc[rb][c][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[rb].p[ta[t]], b.p[tb[t]], acc[rb][c][s], 0, 0,
                                                                            0);
        }
    }
}

template <int PREC, int S, int T>
__global__ __launch_bounds__(256, 2) void k_rho_split(SplitArgs a)
{
    using P = SplitCfg<PREC, S, T>;
    constexpr int NP = P::NP, NPW = P::NPW;
    __shared__ bf8 smem[P::AO_SLOTS + P::C_SLOTS];

    // the MO blocks of a tile follow one another on one XCD
    const int64_t L = logical_block(blockIdx.x, a.nblocks);
    const int mb = (int)(L % a.nb);
    const int64_t tn = L / a.nb;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, n16 = lane & 15;
    // MO tiles of 16 spread evenly over the blocks: T or T - 1 each
    const int q = a.nt / a.nb, rem = a.nt - q * a.nb;
    const int nv = q + (mb < rem ? 1 : 0), m0 = 16 * (mb * q + min(mb, rem));
    const int steps = a.count[tn];

    f4 acc[T][NPW][S];
#pragma unroll
    for (int rb = 0; rb < T; ++rb)
#pragma unroll
        for (int c = 0; c < NPW; ++c)
#pragma unroll
            for (int s = 0; s < S; ++s) acc[rb][c][s] = f4{0.f, 0.f, 0.f, 0.f};
    if (steps > 0) {
        if (nv == T) split_loop<PREC, S, T, T>(a, smem, tn, m0, steps, lane, wave, acc);
        else split_loop<PREC, S, T, T - 1>(a, smem, tn, m0, steps, lane, wave, acc);
    }

    // ---- epilogue: lane holds Phi_s[m0 + 16 rb + 4 g + i][point (wave NPW + c) 16 + n16]
#pragma unroll
    for (int c = 0; c < NPW; ++c) {
        double v[S];
#pragma unroll
        for (int s = 0; s < S; ++s) v[s] = 0.0;
#pragma unroll
        for (int rb = 0; rb < T; ++rb) {
            if (rb >= nv) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double w = a.occ[m0 + 16 * rb + 4 * g + i];
                const double f0 = acc[rb][c][0][i];
                v[0] += w * (f0 * f0);
#pragma unroll
                for (int s = 1; s < S; ++s) v[s] += 2.0 * w * (f0 * (double)acc[rb][c][s][i]);
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            v[s] += __shfl_xor(v[s], 16);
            v[s] += __shfl_xor(v[s], 32);
        }
        const int64_t p = tn * NP + (wave * NPW + c) * 16 + n16;
        if (g == 0 && p < a.np)
#pragma unroll
            for (int s = 0; s < S; ++s) a.partial[((int64_t)mb * S + s) * a.ld + p] = v[s];
    }
}

// C (FP64 [nmo][nao]) -> [octet of rows][plane][mpad][8] bf16, rows in the fused order
__global__ void k_prep_octets(const double* C, int nmo, int nao, int prec, int64_t mpad, int64_t kpad, const int* colmap,
                              void* out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;   // m fastest, then row
    if (i >= mpad * kpad) return;
    const int64_t k = i / mpad, m = i - k * mpad;
    const int src = colmap[k];
    const double v = (m < nmo && src >= 0) ? C[m * nao + src] : 0.0;
    const int npl = prec == OKMI_PREC_BF16X6 ? 3 : 2;
    store_c_split(v, prec, ((k / 8) * npl * mpad + m) * 8 + k % 8, mpad * 8, out);
}

// Live quads of each tile of `np` columns: one wave per tile tests every shell
// against the tile's bounding box (64 at a time), marks the quads its rows lie
// in and writes the mask and the list of the chunks with a marked quad.
struct QuadArgs {
    GridDesc grid;
    BrickMap bm;
    int64_t p0, n;
    int np;
    const ShellRec* shells;    // internal rows
    int nshell, words, nchunk;  // 64-bit mask words and chunks per tile
    int* list;
    int* count;
    unsigned long long* mask;
};

__global__ __launch_bounds__(64) void k_live_quads(QuadArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned int bits[];   // 2 per mask word
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    for (int w = lane; w < 2 * a.words; w += 64) bits[w] = 0;
    double lo[3], hi[3];
    columns_box(a.grid, a.bm, a.p0, a.n, t * a.np, a.np, lane, lo, hi);
    __syncthreads();
    for (int s = lane; s < a.nshell; s += 64) {
        const ShellRec* sh = a.shells + s;
        const double c[3] = {sh->cx, sh->cy, sh->cz};
        double d2 = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double dd = fmax(fmax(lo[d] - c[d], c[d] - hi[d]), 0.0);
            d2 = fma(dd, dd, d2);
        }
        if (!(d2 < sh->rcut2)) continue;   // a tile with no point in the grid has lo > hi: d2 = inf
        const int e = (sh->row0 + sh->nrow - 1) / QR;
        for (int j = sh->row0 / QR; j <= e; ++j) atomicOr(&bits[j >> 5], 1u << (j & 31));
    }
    __syncthreads();
    int base = 0;
    for (int c0 = 0; c0 < a.nchunk; c0 += 64) {   // lane's chunk: byte c of the mask
        const int c = c0 + lane;
        const unsigned q = c < a.nchunk ? bits[c >> 2] >> (8 * (c & 3)) & 0xff : 0;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(q != 0);
        if (q) a.list[t * a.nchunk + base + __builtin_popcountll(m & ((1ull << lane) - 1))] = c << 8 | (int)q;
        base += __builtin_popcountll(m);
    }
    for (int w = lane; w < a.words; w += 64) a.mask[t * a.words + w] = ((unsigned long long)bits[2 * w + 1] << 32) | bits[2 * w];
    if (lane == 0) a.count[t] = base;
}

template <int PREC, int S, int T>
int launch_t(const SplitArgs& a, hipStream_t st)
{
    OkmiProfScope prof("rho_big", st);
    hipLaunchKernelGGL((k_rho_split<PREC, S, T>), dim3((unsigned)a.nblocks), dim3(256), 0, st, a);
    return 0;
}

template <int PREC, int S>
int launch_split(const SplitArgs& a, int t, hipStream_t st)
{
    return t <= 3 ? launch_t<PREC, S, 3>(a, st) : t == 4 ? launch_t<PREC, S, 4>(a, st) : launch_t<PREC, S, 5>(a, st);
}

}  // namespace

int okmi_launch_rho_big_split(OkmiBasis* b, const GridDesc& g, int64_t p0, int64_t np, const double* d_c,
                              const double* d_occ, int nmo, int prec, int S, const int* drv_out, int nout, double* rho,
                              double* delta, int64_t ld_delta, void* ws, size_t ws_bytes, hipStream_t st)
{
    const int npl = prec == OKMI_PREC_BF16X6 ? 3 : 2, NP = S == 1 ? 128 : 64;
    const int64_t kpad = b->nkpad;
    // as few MO blocks as hold five tiles of 16 each, the tiles spread evenly:
    // T or T - 1 per block
    const int nt = (nmo + 15) / 16, nb = (nt + 4) / 5, T = (nt + nb - 1) / nb;
    const int64_t mpad = 16 * (int64_t)nt;
    const int nquad = (int)(kpad / QR), words = (nquad + 63) / 64, nchunk = (int)(kpad / KS);
    const size_t cbytes = a256((size_t)2 * npl * mpad * kpad), obytes = a256(8 * (size_t)mpad);
    const size_t fixed = cbytes + obytes + 255;
    const size_t per_point = (size_t)S * kpad * 4 + (size_t)nb * S * 8;
    const size_t per_tile = (size_t)words * 8 + 4 + (size_t)nchunk * 4;
    if (ws_bytes < fixed + per_point * 64 + per_tile) {   // (the caller's bound is above it)
        okmi_set_error("rho_big: workspace of %zu bytes is too small (need at least %zu)", ws_bytes,
                       fixed + per_point * 64 + per_tile);
        return 1;
    }
    // a whole regular grid is processed in 4x4x4 bricks, otherwise in range order
    BrickMap bm{};
    int64_t total = np;
    if (g.regular && p0 == 0 && np == g.nx * g.ny * g.nz) {
        bm.on = 1;
        bm.nbx = (g.nx + 3) / 4; bm.nby = (g.ny + 3) / 4; bm.nbz = (g.nz + 3) / 4;
        bm.nx = g.nx; bm.ny = g.ny; bm.nz = g.nz;
        total = bm.nbx * bm.nby * bm.nbz * 64;
    }
    // (a workspace without room for a tile of 128 points takes 64 at a time)
    const int64_t fit = (int64_t)((ws_bytes - fixed) / (per_point * NP + per_tile));
    const int64_t ntile = std::max<int64_t>(1, std::min<int64_t>(fit, (total + NP - 1) / NP));
    const int64_t chunk = fit > 0 ? ntile * NP : 64;
    char* w = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
    __bf16* cpl = (__bf16*)w;
    double* occp = (double*)(w + cbytes);
    float* ao = (float*)(w + cbytes + obytes);
    double* part = (double*)(ao + (size_t)S * kpad * chunk);
    unsigned long long* mask = (unsigned long long*)(part + (size_t)nb * S * chunk);
    int* count = (int*)(mask + (size_t)words * ntile);
    int* list = count + ntile;

    hipLaunchKernelGGL(k_prep_octets, dim3((unsigned)((mpad * kpad + 255) / 256)), dim3(256), 0, st, d_c, nmo, b->nao,
                       prec, mpad, kpad, (const int*)b->d_colmap, (void*)cpl);
    // the padding rows of the AO tiles, which no shell writes
    if (okmi_launch_zero_rows_f32(ao, (int)(chunk / 64 * S), kpad * 64, 64, b->d_padrows, b->npadrows, 64, st))
        return 1;
    hipLaunchKernelGGL(k_pad_occ_big, dim3((unsigned)((mpad + 255) / 256)), dim3(256), 0, st, d_occ, nmo, (int)mpad,
                       occp);
    int codes[4];
    for (int s = 0; s < S; ++s) codes[s] = s;
    OutCodes oc{};
    oc.n = nout;
    for (int r = 0; r < nout; ++r) oc.c[r] = drv_out[r];
    // the AO values end in FP32: the screening bound of that arithmetic
    AoLiveMask am{mask, words, NP == 128 ? 1 : 0, b->d_wshells_s};
    am.quads = true;
    am.tile_stride = S * kpad * 64;
    for (int64_t c0 = 0; c0 < total; c0 += chunk) {
        const int64_t n = std::min(total - c0, chunk), nt_pts = (n + NP - 1) / NP;
        if (bm.on) bm.bk0 = c0 / 64;
        QuadArgs qa{};
        qa.grid = g; qa.bm = bm; qa.p0 = p0 + c0; qa.n = n; qa.np = NP;
        qa.shells = b->d_fshells_s; qa.nshell = b->nshell; qa.words = words; qa.nchunk = nchunk;
        qa.list = list; qa.count = count; qa.mask = mask;
        hipLaunchKernelGGL(k_live_quads, dim3((unsigned)nt_pts), dim3(64), (size_t)words * 8, st, qa);
        AoBricks bk{c0 / 64, n / 64, bm.nbx, bm.nby, bm.nbz};
        bk.tile_stride = am.tile_stride;
        int rc = okmi_launch_ao_eval_ex(b, b->d_ishells_s, b->d_fprims_s, g, bm.on ? 0 : p0 + c0, n, bm.on ? &bk : nullptr,
                                        codes, S, OKMI_F32, ao, 64, kpad * 64, st, &am);
        if (rc) return rc;
        SplitArgs a{};
        a.ao = ao; a.kpad = kpad; a.sub = chunk / 64; a.np = n; a.C = cpl; a.mpad = mpad; a.occ = occp; a.partial = part; a.ld = chunk;
        a.nb = nb; a.nt = nt; a.list = list; a.count = count;
        a.nblocks = nb * nt_pts;
        if (prec == OKMI_PREC_BF16X3) rc = S == 1 ? launch_split<OKMI_PREC_BF16X3, 1>(a, T, st)
                                                  : launch_split<OKMI_PREC_BF16X3, 4>(a, T, st);
        else rc = S == 1 ? launch_split<OKMI_PREC_BF16X6, 1>(a, T, st) : launch_split<OKMI_PREC_BF16X6, 4>(a, T, st);
        if (rc) return rc;
        hipLaunchKernelGGL(k_reduce_big, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, part, nb, S, chunk, n, oc,
                           bm.on ? rho : rho + c0, bm.on ? delta : (delta ? delta + c0 : nullptr), ld_delta, bm);
    }
    return okmi_check_launch("rho_big");
}
