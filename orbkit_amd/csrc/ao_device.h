// Per-point evaluation of one contracted Cartesian shell and its
// derivatives, templated on the angular momentum so that every monomial
// index is a compile-time constant (no register indexing, no scratch).
//
// Math (orbkit/c_grid-based.c:38-71, orbkit/c_support.c:28-175): with
// X = x - A_x etc., r2 = X^2+Y^2+Z^2 and radial sums over primitives
//   S0 = sum_p d_p e_p,  S1 = sum_p (-2 a_p) d_p e_p,  S2 = sum_p 4 a_p^2 d_p e_p,
// (e_p = exp(-a_p r2)) a component x^lx y^ly z^lz gives
//   drv 0   : X^lx Y^ly Z^lz S0
//   d/dx    : (lx X^(lx-1) S0 + X^(lx+1) S1) Y^ly Z^lz
//   d2/dx2  : (lx(lx-1) X^(lx-2) S0 + (2lx+1) X^lx S1 + X^(lx+2) S2) Y^ly Z^lz
//   d2/dxdy : X^(lx+1) Y^(ly+1) Z^lz S2 + K S0, K as orbkit/c_support.c:121-168
//             (lowering term only; the reference's mixed-derivative formula,
//             reproduced for parity).
#pragma once
#include "okmi_common.h"

template <int L, typename R>
struct ShellPows {
    R p[3][L + 3];
    __device__ __forceinline__ void init(R X, R Y, R Z)
    {
        p[0][0] = R(1); p[1][0] = R(1); p[2][0] = R(1);
#pragma unroll
        for (int n = 1; n < L + 3; ++n) {
            p[0][n] = p[0][n - 1] * X;
            p[1][n] = p[1][n - 1] * Y;
            p[2][n] = p[2][n - 1] * Z;
        }
    }
};

// monomial with one exponent shifted; exponent < 0 never reaches here
template <int L, typename R>
__device__ __forceinline__ R mono(const ShellPows<L, R>& P, int lx, int ly, int lz)
{
    return P.p[0][lx] * P.p[1][ly] * P.p[2][lz];
}

// value of Cartesian component C (canonical order) for derivative code D
template <int L, int C, int D, typename R>
__device__ __forceinline__ R cart_comp(const ShellPows<L, R>& P, R S0, R S1, R S2)
{
    constexpr int e[3] = {cart_exp(L, C, 0), cart_exp(L, C, 1), cart_exp(L, C, 2)};
    if constexpr (D == 0) {
        return mono<L, R>(P, e[0], e[1], e[2]) * S0;
    } else if constexpr (D <= 3) {
        constexpr int a = D - 1;
        constexpr int u0 = e[0] + (a == 0), u1 = e[1] + (a == 1), u2 = e[2] + (a == 2);
        R v = mono<L, R>(P, u0, u1, u2) * S1;
        if constexpr (e[a] > 0) {
            constexpr int d0 = e[0] - (a == 0), d1 = e[1] - (a == 1), d2 = e[2] - (a == 2);
            v += R(e[a]) * mono<L, R>(P, d0, d1, d2) * S0;
        }
        return v;
    } else if constexpr (D <= 6) {
        constexpr int a = D - 4;
        constexpr int u0 = e[0] + 2 * (a == 0), u1 = e[1] + 2 * (a == 1), u2 = e[2] + 2 * (a == 2);
        R v = mono<L, R>(P, u0, u1, u2) * S2 + R(2 * e[a] + 1) * mono<L, R>(P, e[0], e[1], e[2]) * S1;
        if constexpr (e[a] >= 2) {
            constexpr int d0 = e[0] - 2 * (a == 0), d1 = e[1] - 2 * (a == 1), d2 = e[2] - 2 * (a == 2);
            v += R(e[a] * (e[a] - 1)) * mono<L, R>(P, d0, d1, d2) * S0;
        }
        return v;
    } else {   // 7: xy, 8: xz, 9: yz
        constexpr int i = D == 9 ? 1 : 0;
        constexpr int j = D == 7 ? 1 : 2;
        constexpr int u0 = e[0] + (i == 0) + (j == 0), u1 = e[1] + (i == 1) + (j == 1), u2 = e[2] + (i == 2) + (j == 2);
        R v = mono<L, R>(P, u0, u1, u2) * S2;
        if constexpr (e[i] == 0 && e[j] > 0) {
            constexpr int d0 = e[0] - (j == 0), d1 = e[1] - (j == 1), d2 = e[2] - (j == 2);
            v += R(e[j]) * mono<L, R>(P, d0, d1, d2) * S0;
        } else if constexpr (e[i] > 0 && e[j] == 0) {
            constexpr int d0 = e[0] - (i == 0), d1 = e[1] - (i == 1), d2 = e[2] - (i == 2);
            v += R(e[i]) * mono<L, R>(P, d0, d1, d2) * S0;
        } else if constexpr (e[i] > 0 && e[j] > 0) {
            constexpr int d0 = e[0] - (i == 0) - (j == 0), d1 = e[1] - (i == 1) - (j == 1),
                          d2 = e[2] - (i == 2) - (j == 2);
            v += R(e[i] * e[j]) * mono<L, R>(P, d0, d1, d2) * S0;
        }
        return v;
    }
}

template <int L, int D, typename R, int C = 0>
__device__ __forceinline__ void cart_all(const ShellPows<L, R>& P, R S0, R S1, R S2, R* out)
{
    if constexpr (C < ncart(L)) {
        out[C] = cart_comp<L, C, D, R>(P, S0, S1, S2);
        cart_all<L, D, R, C + 1>(P, S0, S1, S2, out);
    }
}

// canonical index of component (lx, ly, lz) of angular momentum l
__host__ __device__ constexpr int cart_index(int l, int lx, int ly, int lz)
{
    for (int c = 0; c < ncart(l); ++c)
        if (cart_exp(l, c, 0) == lx && cart_exp(l, c, 1) == ly && cart_exp(l, c, 2) == lz) return c;
    return -1;
}

// Value and first derivatives of all components from shared monomials:
//   chi_c = m_c S0,   d_a chi_c = (R_a S1) m_c + e_a (m_{c - 1_a} S0),
// m_c the degree-L monomial of component c, m_{c - 1_a} the degree-(L-1)
// one with exponent a lowered (the same terms as cart_comp, D = 0..3,
// evaluated once per shell and point instead of once per derivative).
template <int L, int C, typename R>
__device__ __forceinline__ void first_mono(const ShellPows<L, R>& P, R* m)
{
    if constexpr (C < ncart(L)) {
        m[C] = mono<L, R>(P, cart_exp(L, C, 0), cart_exp(L, C, 1), cart_exp(L, C, 2));
        first_mono<L, C + 1, R>(P, m);
    }
}

template <int L, int C, typename R>
__device__ __forceinline__ void lower_mono(const ShellPows<L, R>& P, R S0, R* u)
{
    if constexpr (L > 0 && C < ncart(L - 1)) {
        u[C] = mono<L, R>(P, cart_exp(L - 1, C, 0), cart_exp(L - 1, C, 1), cart_exp(L - 1, C, 2)) * S0;
        lower_mono<L, C + 1, R>(P, S0, u);
    }
}

// out[c] = d_a chi_c for axis A, with RS1 = R_a S1
template <int L, int A, int C, typename R>
__device__ __forceinline__ void first_deriv(const R* m, const R* u, R RS1, R* out)
{
    if constexpr (C < ncart(L)) {
        constexpr int e0 = cart_exp(L, C, 0), e1 = cart_exp(L, C, 1), e2 = cart_exp(L, C, 2);
        constexpr int ea = A == 0 ? e0 : A == 1 ? e1 : e2;
        if constexpr (ea > 0) {
            constexpr int lo = cart_index(L - 1, e0 - (A == 0), e1 - (A == 1), e2 - (A == 2));
            out[C] = fma(RS1, m[C], R(ea) * u[lo]);
        } else {
            out[C] = RS1 * m[C];
        }
        first_deriv<L, A, C + 1, R>(m, u, RS1, out);
    }
}

// sum_c w_c e_a(c) u_{c - 1_a} for axis A, u the degree-(L-1) monomials
// (times S0): the lowered-exponent half of sum_c w_c d_a chi_c
template <int L, int A, int C, typename R>
__device__ __forceinline__ R lowered_dot(const R* w, const R* u, R acc)
{
    if constexpr (C < ncart(L)) {
        constexpr int e0 = cart_exp(L, C, 0), e1 = cart_exp(L, C, 1), e2 = cart_exp(L, C, 2);
        constexpr int ea = A == 0 ? e0 : A == 1 ? e1 : e2;
        if constexpr (ea > 0) {
            constexpr int lo = cart_index(L - 1, e0 - (A == 0), e1 - (A == 1), e2 - (A == 2));
            acc = fma(w[C] * R(ea), u[lo], acc);
        }
        return lowered_dot<L, A, C + 1, R>(w, u, acc);
    } else {
        return acc;
    }
}

// runtime (wave-uniform) derivative code -> compile-time evaluation
template <int L, typename R>
__device__ __forceinline__ void cart_drv(const ShellPows<L, R>& P, int d, R S0, R S1, R S2, R* out)
{
    switch (d) {
    case 0: cart_all<L, 0, R>(P, S0, S1, S2, out); break;
    case 1: cart_all<L, 1, R>(P, S0, S1, S2, out); break;
    case 2: cart_all<L, 2, R>(P, S0, S1, S2, out); break;
    case 3: cart_all<L, 3, R>(P, S0, S1, S2, out); break;
    case 4: cart_all<L, 4, R>(P, S0, S1, S2, out); break;
    case 5: cart_all<L, 5, R>(P, S0, S1, S2, out); break;
    case 6: cart_all<L, 6, R>(P, S0, S1, S2, out); break;
    case 7: cart_all<L, 7, R>(P, S0, S1, S2, out); break;
    case 8: cart_all<L, 8, R>(P, S0, S1, S2, out); break;
    default: cart_all<L, 9, R>(P, S0, S1, S2, out); break;
    }
}

// a b + c.  A compile-time constant c goes in a scalar register pair of one
// v_fma_f64: left to itself the compiler takes the two-operand form for a
// polynomial step and copies the coefficient into its result first, two
// vector instructions per coefficient.
__device__ __forceinline__ double fma_coef(double a, double b, double c)
{
    if (__builtin_constant_p(c)) {
        double d;
        asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
        return d;
    }
    return fma(a, b, c);
}

// exp(-t) in FP64 for t >= 0: Cody-Waite reduction -t = s - k ln2, |s| <= ln2/2
// (ln2 in a high part exact in 32 bits and a low part; r without the low part is
// exact), exp(s) as 1 + s + s^2 R(s) with R from the Chebyshev interpolant of
// degree 11 on that interval (relative error below 2e-17), and 2^-k by exponent
// adjustment, which underflows to +0.  1 + s is formed as h = 1 + r and what h
// and the low part leave out, so that the last addition makes most of the error:
// at most 0.79 ulp, 0.252 on average (the device library's exp: 0.87 and 0.256;
// 1 + (s + s^2 R) would give 1.13 and 0.264 with four operations less).  Even and
// odd coefficients run in two chains: most shells have one primitive in reach of
// a tile, so the chain of its exponential is what a wave waits for.  Branch-free:
// t is clamped to 1e4 (+0 in FP64).
__device__ __forceinline__ double gauss_f64(double t)
{
    t = fmin(t, 1.0e4);
    const double k = __builtin_rint(t * 1.4426950408889634);
    const double r = fma(k, 6.93147180369123816490e-01, -t);
    const double s = fma(k, 1.90821492927058770002e-10, r);
    const double h = 1.0 + r, l = fma(k, 1.90821492927058770002e-10, r - (h - 1.0));
    const double q = s * s;
    double e = fma_coef(q, 2.763263963904103e-07, 2.4801485482328494e-05);
    double o = fma_coef(q, 2.5110037605963777e-08, 2.755724091857897e-06);
    e = fma_coef(e, q, 0.0013888888952314775);
    o = fma_coef(o, q, 0.00019841269890047113);
    e = fma_coef(e, q, 0.0416666666664881);
    o = fma_coef(o, q, 0.008333333333319601);
    e = fma_coef(e, q, 0.5000000000000019);
    o = fma_coef(o, q, 0.1666666666666668);
    return ldexp(h + fma(q, fma(o, s, e), l), -(int)k);
}

// exp(-t) to FP32 accuracy for any t >= 0 given in FP64: the range reduction
// t*log2(e) = n + f (n integer, 0 <= f < 1) is done in FP64 so that large
// arguments (tight exponents far from their centre) keep a full FP32
// mantissa; 2^-f uses the hardware exp2 (v_exp_f32) and 2^-n an exponent
// adjustment.  Results below FP32's range flush to +0.
__device__ __forceinline__ float gauss_f32(double t)
{
    const double u = t * 1.4426950408889634;   // log2(e)
    if (u >= 150.0) return 0.0f;
    const double n = floor(u);
    const float f = (float)(u - n);
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(-f), -(int)n);
}

// exp(-t) for t >= 0 in FP64 with 2.6e-9 relative error (under 1/20 of an
// FP32 half-ulp), for the paths whose AO values end in FP32 or narrower.
// Cody-Waite reduction t = k ln2 + r, |r| <= ln2/2 (ln2 split in a high part
// exact in 32 bits and a low part), then exp(s), s = -r, by a degree-6
// polynomial: the Chebyshev interpolant of exp on [-ln2/2, ln2/2] (7
// Chebyshev nodes, converted to monomial coefficients), and 2^-k by exponent
// adjustment, which underflows to +0 for large t.  Branch-free: t is
// clamped to 1e4 (exp(-1e4) is +0 in FP64).
__device__ __forceinline__ double gauss_f64_fast(double t)
{
    t = fmin(t, 1.0e4);
    const double k = __builtin_rint(t * 1.4426950408889634);
    double r = fma(-k, 6.93147180369123816490e-01, t);
    r = fma(-k, 1.90821492927058770002e-10, r);
    const double s = -r;
    const auto fma = fma_coef;
    double p = 0.0013941118940759135;
    p = fma(p, s, 0.0083751347746787615);
    p = fma(p, s, 0.041666352770387056);
    p = fma(p, s, 0.16666415414041169);
    p = fma(p, s, 0.50000000471463202);
    p = fma(p, s, 1.0000000377388703);
    p = fma(p, s, 0.99999999999999989);
    return ldexp(p, -(int)k);
}

// Standard real-solid-harmonic rows in orbkit's (l, m) order
// (m = 0, 1, -1, 2, -2, ...; p: x, y, z), each as at most three canonical
// Cartesian components with orbkit's cart2sph coefficient (orbkit/tools.py:
// 148-191) times the 1/sqrt((2lx-1)!!(2ly-1)!!(2lz-1)!!) normalisation
// factor.  basis_create checks each spherical shell's transform against this
// table before it is evaluated through it.
struct SphTerm { int c; double v; };
struct SphRow { int n; SphTerm t[3]; };
__host__ __device__ constexpr SphRow sph_row(int l, int r)
{
    constexpr SphRow L0[1] = {{1, {{0, 1.0}, {0, 0.0}, {0, 0.0}}}};
    constexpr SphRow L1[3] = {{1, {{0, 1.0}, {0, 0.0}, {0, 0.0}}},
                              {1, {{1, 1.0}, {0, 0.0}, {0, 0.0}}},
                              {1, {{2, 1.0}, {0, 0.0}, {0, 0.0}}}};
    constexpr SphRow L2[5] = {{3, {{0, -0.28867513459481292}, {1, -0.28867513459481292}, {2, 0.57735026918962584}}},
                              {1, {{4, 1.0}, {0, 0.0}, {0, 0.0}}},
                              {1, {{5, 1.0}, {0, 0.0}, {0, 0.0}}},
                              {2, {{0, 0.5}, {1, -0.5}, {0, 0.0}}},
                              {1, {{3, 1.0}, {0, 0.0}, {0, 0.0}}}};
    constexpr SphRow L3[7] = {{3, {{2, 0.2581988897471611}, {5, -0.3872983346207417}, {8, -0.3872983346207417}}},
                              {3, {{0, -0.15811388300841897}, {3, -0.15811388300841897}, {6, 0.63245553203367599}}},
                              {3, {{1, -0.15811388300841897}, {4, -0.15811388300841897}, {7, 0.63245553203367599}}},
                              {2, {{5, 0.5}, {8, -0.5}, {0, 0.0}}},
                              {1, {{9, 1.0}, {0, 0.0}, {0, 0.0}}},
                              {2, {{0, 0.20412414523193148}, {3, -0.61237243569579447}, {0, 0.0}}},
                              {2, {{1, -0.20412414523193148}, {4, 0.61237243569579447}, {0, 0.0}}}};
    return l == 0 ? L0[r] : l == 1 ? L1[r] : l == 2 ? L2[r] : L3[r];
}

// Output rows of a standard spherical shell (sph_row table) or a standard
// Cartesian shell (component norm factors) from the canonical Cartesian
// values c, unrolled at compile time: store(r, value) for each row r.
template <int L, int R, typename Store>
__device__ __forceinline__ void sph_rows_to(const double* c, Store&& store)
{
    if constexpr (L <= 3 && R < 2 * L + 1) {
        constexpr SphRow row = sph_row(L, R);
        double v = row.t[0].v * c[row.t[0].c];
        if constexpr (row.n > 1) v = fma(row.t[1].v, c[row.t[1].c], v);
        if constexpr (row.n > 2) v = fma(row.t[2].v, c[row.t[2].c], v);
        store(R, v);
        sph_rows_to<L, R + 1>(c, store);
    }
}

// 1/sqrt((2lx-1)!!(2ly-1)!!(2lz-1)!!) of canonical component c
__host__ __device__ constexpr double cart_norm(int l, int c)
{
    int d = 1;
    for (int a = 0; a < 3; ++a) {
        int e = cart_exp(l, c, a);
        for (int n = 2 * e - 1; n > 0; n -= 2) d *= n;
    }
    return d == 1 ? 1.0 : d == 3 ? 0.57735026918962584 : d == 9 ? 0.33333333333333333
         : d == 15 ? 0.2581988897471611 : d == 105 ? 0.09759000729485333 : 0.0;
}

template <int L, int R, typename Store>
__device__ __forceinline__ void cart_rows_to(const double* c, Store&& store)
{
    if constexpr (R < ncart(L)) {
        store(R, c[R] * cart_norm(L, R));
        cart_rows_to<L, R + 1>(c, store);
    }
}

// Rows of a standard spherical (sph_row) or Cartesian (component norms)
// shell straight from the monomials, instead of the Cartesian values of each
// AO set first and their combinations after: with row polynomial
// P = sum_t v_t m_t of the degree-L monomials,
//   chi = P S0,  d_a chi = P (R_a S1) + (d_a P) S0,
//   d_aa chi = P (S1 + R_a^2 S2) + (d_a P) (2 R_a S1) + (d_aa P) S0.
template <int L, bool SPH> __host__ __device__ constexpr int shell_rows() { return SPH ? 2 * L + 1 : ncart(L); }
template <int L, bool SPH, int R> __host__ __device__ constexpr SphRow shell_row()
{
    if constexpr (SPH) return sph_row(L, R);
    else return SphRow{1, {{R, cart_norm(L, R)}, {0, 0.0}, {0, 0.0}}};
}

// Row polynomials of a shell at one point.  Standard spherical d and f rows
// (sph_row's coefficients) in factored form from the quadratic monomials
// (fewer operations and registers than the ten cubic ones); other rows from
// the degree-L monomials.
template <int L, bool SPH> struct RowPolys {
    double m[ncart(L)];
    __device__ __forceinline__ RowPolys(double X, double Y, double Z)
    {
        ShellPows<L, double> P;
        P.init(X, Y, Z);
        first_mono<L, 0, double>(P, m);
    }
    template <int R> __device__ __forceinline__ double row() const
    {
        constexpr SphRow row = shell_row<L, SPH, R>();
        double v = row.t[0].v == 1.0 ? m[row.t[0].c] : row.t[0].v * m[row.t[0].c];
        if constexpr (row.n > 1) v = fma(row.t[1].v, m[row.t[1].c], v);
        if constexpr (row.n > 2) v = fma(row.t[2].v, m[row.t[2].c], v);
        return v;
    }
};
template <> struct RowPolys<2, true> {
    double X, Y, Z;
    __device__ __forceinline__ RowPolys(double x, double y, double z) : X(x), Y(y), Z(z) {}
    template <int R> __device__ __forceinline__ double row() const
    {
        constexpr double q = sph_row(2, 0).t[2].v;   // 1 / sqrt(3); x^2 + y^2 has -q/2
        if constexpr (R == 0) return q * fma(Z, Z, -0.5 * fma(X, X, Y * Y));
        if constexpr (R == 1) return X * Z;
        if constexpr (R == 2) return Y * Z;
        if constexpr (R == 3) return 0.5 * (X - Y) * (X + Y);
        return X * Y;
    }
};
template <> struct RowPolys<3, true> {
    double X, Y, Z;
    __device__ __forceinline__ RowPolys(double x, double y, double z) : X(x), Y(y), Z(z) {}
    template <int R> __device__ __forceinline__ double row() const
    {
        constexpr double a0 = sph_row(3, 0).t[0].v, a1 = sph_row(3, 1).t[2].v, a5 = sph_row(3, 5).t[0].v;
        if constexpr (R == 0) return a0 * (Z * fma(Z, Z, -1.5 * fma(X, X, Y * Y)));
        if constexpr (R == 1) return a1 * (X * fma(Z, Z, -0.25 * fma(X, X, Y * Y)));
        if constexpr (R == 2) return a1 * (Y * fma(Z, Z, -0.25 * fma(X, X, Y * Y)));
        if constexpr (R == 3) return 0.5 * Z * ((X - Y) * (X + Y));
        if constexpr (R == 4) return X * Y * Z;
        if constexpr (R == 5) return a5 * (X * fma(X, X, -3.0 * (Y * Y)));
        return a5 * (Y * fma(3.0 * X, X, -(Y * Y)));
    }
};

// acc + sum over the row's terms of v_t e (e - 1) ... (N factors of axis A's
// exponent) u[component with that exponent lowered by N]; u: the degree
// L - N monomials (times a radial sum)
template <int L, bool SPH, int R, int A, int N, int T = 0>
__device__ __forceinline__ double row_lowered(const double* u, double acc)
{
    constexpr SphRow row = shell_row<L, SPH, R>();
    if constexpr (T < row.n) {
        constexpr int c = row.t[T].c;
        constexpr int e[3] = {cart_exp(L, c, 0), cart_exp(L, c, 1), cart_exp(L, c, 2)};
        if constexpr (e[A] >= N) {
            constexpr double f = row.t[T].v * (N == 1 ? e[A] : e[A] * (e[A] - 1));
            constexpr int lo = cart_index(L - N, e[0] - N * (A == 0), e[1] - N * (A == 1), e[2] - N * (A == 2));
            acc = f == 1.0 ? acc + u[lo] : fma(f, u[lo], acc);
        }
        return row_lowered<L, SPH, R, A, N, T + 1>(u, acc);
    } else {
        return acc;
    }
}

// the degree-L monomials times f
template <int L, int C = 0>
__device__ __forceinline__ void scaled_monos(double X, double Y, double Z, double f, double* u)
{
    if constexpr (L >= 0) {
        ShellPows<(L > 0 ? L : 0), double> P;
        P.init(X, Y, Z);
        first_mono<(L > 0 ? L : 0), 0, double>(P, u);
#pragma unroll
        for (int c = 0; c < ncart(L > 0 ? L : 0); ++c) u[c] *= f;
    }
}

// The AO sets of one pass (PassCodes) of each row of a standard shell
template <int L, bool SPH, int PASS> struct RowSets {
    static constexpr int NS = PASS == 0 ? 1 : PASS == 4 ? 7 : 4;
    RowPolys<L, SPH> m;
    double S0, R1[3], R2[3];
    double u1[L > 0 ? ncart(L - 1) : 1];                 // degree L - 1 monomials (PASS 1: times S0)
    double u2[PASS >= 2 && L > 1 ? ncart(L - 2) : 1];    // degree L - 2 monomials times S0
    ShellPows<L, double> P;                              // PASS 3
    double s1, s2;

    __device__ __forceinline__ RowSets(double X, double Y, double Z, double s0_, double s1_, double s2_)
        : m(X, Y, Z), S0(s0_), s1(s1_), s2(s2_)
    {
        if constexpr (PASS == 1 || PASS == 2 || PASS == 4) {
            R1[0] = X * s1_;
            R1[1] = Y * s1_;
            R1[2] = Z * s1_;
            scaled_monos<L - 1>(X, Y, Z, PASS == 1 ? s0_ : 1.0, u1);
        }
        if constexpr (PASS == 2 || PASS == 4) {
            R2[0] = fma(X * X, s2_, s1_);
            R2[1] = fma(Y * Y, s2_, s1_);
            R2[2] = fma(Z * Z, s2_, s1_);
            scaled_monos<L - 2>(X, Y, Z, s0_, u2);
        }
        if constexpr (PASS == 3) P.init(X, Y, Z);
    }
    template <int R, int D, int T = 0> __device__ __forceinline__ double mixed(double acc) const
    {
        constexpr SphRow row = shell_row<L, SPH, R>();
        if constexpr (T < row.n) {
            return mixed<R, D, T + 1>(fma(row.t[T].v, cart_comp<L, row.t[T].c, D, double>(P, S0, s1, s2), acc));
        } else {
            return acc;
        }
    }
    // d_aa of the row: p its polynomial, d its derivative along axis A
    template <int R, int A> __device__ __forceinline__ double second(double p, double d) const
    {
        return fma(d, 2.0 * R1[A], row_lowered<L, SPH, R, A, 2>(u2, p * R2[A]));
    }
    template <int R> __device__ __forceinline__ void row(double (&v)[NS]) const
    {
        const double p = m.template row<R>();
        v[0] = p * S0;
        if constexpr (PASS == 1) {
            v[1] = row_lowered<L, SPH, R, 0, 1>(u1, p * R1[0]);
            v[2] = row_lowered<L, SPH, R, 1, 1>(u1, p * R1[1]);
            v[3] = row_lowered<L, SPH, R, 2, 1>(u1, p * R1[2]);
        } else if constexpr (PASS == 2 || PASS == 4) {
            const double d[3] = {row_lowered<L, SPH, R, 0, 1>(u1, 0.0), row_lowered<L, SPH, R, 1, 1>(u1, 0.0),
                                 row_lowered<L, SPH, R, 2, 1>(u1, 0.0)};
            if constexpr (PASS == 4) {
                v[1] = fma(d[0], S0, p * R1[0]);
                v[2] = fma(d[1], S0, p * R1[1]);
                v[3] = fma(d[2], S0, p * R1[2]);
            }
            v[NS - 3] = second<R, 0>(p, d[0]);
            v[NS - 2] = second<R, 1>(p, d[1]);
            v[NS - 1] = second<R, 2>(p, d[2]);
        } else if constexpr (PASS == 3) {
            v[1] = mixed<R, 7>(0.0);
            v[2] = mixed<R, 8>(0.0);
            v[3] = mixed<R, 9>(0.0);
        }
    }
};

// f(row, values of the sets) for every row from R on
template <int R, int L, bool SPH, int PASS, typename F>
__device__ __forceinline__ void each_row(const RowSets<L, SPH, PASS>& rows, F&& f)
{
    if constexpr (R < shell_rows<L, SPH>()) {
        double v[RowSets<L, SPH, PASS>::NS];
        rows.template row<R>(v);
        f(R, v);
        each_row<R + 1>(rows, f);
    }
}
