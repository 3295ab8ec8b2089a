// sdbe_pfb_solve.hpp -- per-branch arithmetic of the PFB inverse's
// constant-coefficient solve (sdbe_pfb.hip): the minimum-phase factor, a plan's
// tables, the rule that admits a plan, and the rank-3 corner.  Plain functions of
// one branch, host and device, so that the accuracy of the solve and of the rule
// can be checked without a GPU.
//
// P P^T is Toeplitz per branch, so it has a constant minimum-phase factor b:
// b(q) = b0 + b1 q + b2 q^2 + b3 q^3 with the taps' autocorrelation and no zero
// inside the unit circle (the taps' polynomial with its zeros inside reflected),
// and with B the lower-triangular Toeplitz matrix of b
//   P P^T = B B^T + E H H^T E^T,   H[i][m] = b_{i+m+1}  (E: the first three rows).
// B B^T is two recursive filters with three constant coefficients beta = b_k / b0,
// and the corner is a rank-3 correction of the first three right-hand sides by
// g = H t, t = H^T (first three rows of the solution).  In scaled units
// v = b0 B^-1 y, zeta = b0^2 z:
//   v_i = y_i - beta1 v_{i-1} - beta2 v_{i-2} - beta3 v_{i-3},
//   zeta_i = v_i - beta1 zeta_{i+1} - beta2 zeta_{i+2} - beta3 zeta_{i+3},
// and t is iterated: t += S^-1 (H^T zeta(t) - t), S = I + H^T G H, G the first 3 x 3
// block of (B B^T)^-1.  S is symmetric with no eigenvalue below 1, and the
// iteration only needs it to a few digits: what the solution satisfies in the end is
// the equation of t with the filters' own zeta.
#pragma once

#include <math.h>
#include <stddef.h>

namespace sdbe {
namespace pfb {

constexpr int SR = 32, SWV = 8, SBLK = SR * SWV;     // rows per span, spans and rows per block
// rows of a plan's table, one double per branch each
constexpr int TB_BETA = 0;                // beta1..3
constexpr int TB_WZ = 3;                  // taps / b0^2
constexpr int TB_CS = 7;                  // C^32: the state after a span of no input
constexpr int TB_CB = 16;                 // C^256
constexpr int TB_RB = 25;                 // a block's head zeta per unit incoming state
constexpr int TB_HB = 34;                 // its impulse response h251..h255
constexpr int TB_GB = 39;                 // G of 256 rows
constexpr int TB_N = 48;

// Double-double arithmetic (Dekker's product by FMA, Knuth's sum): h + l, |l| at
// most half an ulp of h.  No contraction of the plain operations: fusing the
// product into the sum that follows it would count its rounding error twice.
struct Dd {
    double h = 0.0, l = 0.0;
};
__host__ __device__ __forceinline__ Dd dd_norm(double h, double l) {
#pragma clang fp contract(off)
    const double s = h + l;
    return Dd{s, l - (s - h)};
}
__host__ __device__ __forceinline__ Dd dd_add(Dd a, Dd b) {
#pragma clang fp contract(off)
    const double s = a.h + b.h, t = s - a.h;
    return dd_norm(s, (a.h - (s - t)) + (b.h - t) + (a.l + b.l));
}
__host__ __device__ __forceinline__ Dd dd_neg(Dd a) { return Dd{-a.h, -a.l}; }
__host__ __device__ __forceinline__ Dd dd_mul(Dd a, Dd b) {
#pragma clang fp contract(off)
    const double p = a.h * b.h;
    return dd_norm(p, fma(a.h, b.h, -p) + fma(a.h, b.l, a.l * b.h));
}
// a - b c
__host__ __device__ __forceinline__ Dd dd_sub_mul(Dd a, Dd b, Dd c) { return dd_add(a, dd_neg(dd_mul(b, c))); }
// The quotient of the leading parts, corrected twice by the remainder.
__host__ __device__ __forceinline__ Dd dd_div(Dd a, Dd b) {
#pragma clang fp contract(off)
    const double q0 = a.h / b.h;
    const Dd r0 = dd_sub_mul(a, b, Dd{q0, 0.0});
    const double q1 = r0.h / b.h;
    const Dd r1 = dd_sub_mul(r0, b, Dd{q1, 0.0});
    return dd_add(dd_norm(q0, q1), Dd{r1.h / b.h, 0.0});
}
// One Newton step on the root of the leading part.
__host__ __device__ __forceinline__ Dd dd_sqrt(Dd a) {
    const double s = sqrt(a.h);
    if (!(s > 0.0)) return Dd{0.0, 0.0};
    const Dd r = dd_sub_mul(a, Dd{s, 0.0}, Dd{s, 0.0});
    return dd_norm(s, 0.5 * r.h / s);
}
__host__ __device__ __forceinline__ Dd dd(double x) { return Dd{x, 0.0}; }

// The minimum-phase factor b of the taps w.  The taps' cubic (in the order with
// the larger end coefficient first) gives up its real zero -- Cardano's formula,
// then Newton steps -- by deflation from the end that keeps the remaining
// coefficients accurate; then the quadratic; zeros outside the unit circle are
// reflected.  In double-double: b's autocorrelation has to be the taps' to FP64's
// last digit, because zeros together near the circle amplify any difference as
// the condition of P P^T does (FP64 throughout was off by 1e-13 there, which lost up
// to three digits of the result).
__host__ __device__ inline void min_phase(const double (&w)[4], Dd (&b)[4]) {
    const bool rev = fabs(w[3]) > fabs(w[0]);
    const double c[4] = {rev ? w[3] : w[0], rev ? w[2] : w[1], rev ? w[1] : w[2], rev ? w[0] : w[3]};
    for (int i = 0; i < 4; ++i) b[i] = dd(0.0);
    if (c[0] == 0.0) {              // both ends vanish: two taps
        const bool f = fabs(c[1]) >= fabs(c[2]);
        b[0] = dd(f ? c[1] : c[2]);
        b[1] = dd(f ? c[2] : c[1]);
        return;
    }
    const Dd A = dd_div(dd(c[1]), dd(c[0])), B = dd_div(dd(c[2]), dd(c[0])), C = dd_div(dd(c[3]), dd(c[0]));
    double x;
    {
        const double a = A.h, Q = (a * a - 3.0 * B.h) / 9.0, R = (2.0 * a * a * a - 9.0 * a * B.h + 27.0 * C.h) / 54.0;
        if (R * R < Q * Q * Q) {    // three real zeros: the largest
            const double th = acos(fmax(-1.0, fmin(1.0, R / sqrt(Q * Q * Q))));
            const double m = -2.0 * sqrt(Q), tau = 6.283185307179586476925286766559;
            x = m * cos(th / 3.0) - a / 3.0;
            for (int k = 1; k < 3; ++k) {
                const double y = m * cos((th + k * tau) / 3.0) - a / 3.0;
                if (fabs(y) > fabs(x)) x = y;
            }
        } else {
            const double s = -copysign(cbrt(fabs(R) + sqrt(fmax(R * R - Q * Q * Q, 0.0))), R);
            x = s + (s != 0.0 ? Q / s : 0.0) - a / 3.0;
        }
    }
    Dd r = dd(x);
    auto value = [&](Dd y) { return dd_add(dd_mul(dd_add(dd_mul(dd_add(y, A), y), B), y), C); };
    Dd f = value(r);
    for (int k = 0; k < 64; ++k) {      // a triple zero converges by 2/3 a step
        const Dd d = dd_add(dd_mul(dd_add(dd_mul(dd(3.0), r), dd_mul(dd(2.0), A)), r), B);
        if (d.h == 0.0 || f.h == 0.0) break;
        const Dd y = dd_add(r, dd_neg(dd_div(f, d))), g = value(y);
        if (!(fabs(g.h) < fabs(f.h))) break;
        r = y;
        f = g;
    }
    // x^2 + d1 x + d0: coefficients above the largest of the terms |C|, |B r|,
    // |A r^2|, |r^3| from the top, those below it from the bottom
    Dd d1 = dd_add(A, r), d0 = dd_add(B, dd_mul(d1, r));
    if (r.h != 0.0) {
        const double q = r.h, t0 = fabs(C.h), t1 = fabs(B.h * q), t2 = fabs(A.h * q * q), t3 = fabs(q * q * q);
        if (fmax(t2, t3) > fmax(t0, t1) || t1 > t0) d0 = dd_neg(dd_div(C, r));
        if (fmax(t2, t3) > fmax(t0, t1)) d1 = dd_div(dd_add(d0, dd_neg(B)), r);
    }
    Dd p[4] = {dd(c[0]), dd(0.0), dd(0.0), dd(0.0)};
    bool any = false;                   // a zero was reflected
    auto outside = [](Dd y) { return fabs(y.h) > 1.0 || (fabs(y.h) == 1.0 && y.h * y.l > 0.0); };
    auto times = [&](Dd y) {            // times (x - y), or reflected: (1 - x y)
        const bool out = outside(y);
        any = any || out;
        const Dd u = out ? dd_neg(y) : dd(1.0), v = out ? dd(1.0) : dd_neg(y);
        for (int i = 3; i >= 1; --i) p[i] = dd_add(dd_mul(p[i], u), dd_mul(p[i - 1], v));
        p[0] = dd_mul(p[0], u);
    };
    times(r);
    const Dd disc = dd_sub_mul(dd_mul(d1, d1), dd(4.0), d0);
    if (disc.h >= 0.0) {
        const Dd q = dd_sqrt(disc), s = dd_mul(dd(-0.5), dd_add(d1, d1.h < 0.0 ? dd_neg(q) : q));
        times(s);
        times(s.h != 0.0 ? dd_div(d0, s) : dd(0.0));
    } else {
        const bool out = d0.h > 1.0;
        any = any || out;
        const Dd e0 = out ? d0 : dd(1.0), e2 = out ? dd(1.0) : d0, p0 = p[0], p1 = p[1];
        p[0] = dd_mul(p0, e0);
        p[1] = dd_add(dd_mul(p0, d1), dd_mul(p1, e0));
        p[2] = dd_add(dd_mul(p0, e2), dd_mul(p1, d1));
        p[3] = dd_mul(p1, e2);
    }
    // taps that are minimum phase already (in either order) are the factor, exactly
    for (int i = 0; i < 4; ++i) b[i] = any ? p[i] : dd(c[i]);
}

// 3 x 3 matrices, m[3 r + c]: o = a b, and o = a b^T
__host__ __device__ __forceinline__ void mat_mul(double (&o)[9], const double (&a)[9], const double (&b)[9]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            o[3 * r + c] = fma(a[3 * r], b[c], fma(a[3 * r + 1], b[3 + c], a[3 * r + 2] * b[6 + c]));
}
__host__ __device__ __forceinline__ void mat_mul_t(double (&o)[9], const double (&a)[9], const double (&b)[9]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            o[3 * r + c] = fma(a[3 * r], b[3 * c], fma(a[3 * r + 1], b[3 * c + 1], a[3 * r + 2] * b[3 * c + 2]));
}

// G of m blocks of 256 rows and P = C^(256 m), from one block's G and C, by
// doubling over the bits of m.
__host__ __device__ inline void block_gram(int m, const double (&CB)[9], const double (&GB)[9], double (&P)[9],
                                           double (&G)[9]) {
    double t[9], u[9];
    auto add = [&](const double (&X)[9]) {        // G += P X P^T
        mat_mul(t, P, X);
        mat_mul_t(u, t, P);
        for (int i = 0; i < 9; ++i) G[i] += u[i];
    };
    for (int i = 0; i < 9; ++i) {
        P[i] = CB[i];
        G[i] = GB[i];
    }
    int top = 0;
    while ((m >> (top + 1)) != 0) ++top;
    for (int bit = top - 1; bit >= 0; --bit) {
        double s[9];
        for (int i = 0; i < 9; ++i) s[i] = G[i];
        add(s);
        mat_mul(t, P, P);
        for (int i = 0; i < 9; ++i) P[i] = t[i];
        if ((m >> bit) & 1) {
            add(GB);
            mat_mul(t, CB, P);
            for (int i = 0; i < 9; ++i) P[i] = t[i];
        }
    }
}

struct V3 {
    double a, b, c;
};
__host__ __device__ __forceinline__ V3 v3_add(V3 x, V3 y) { return V3{x.a + y.a, x.b + y.b, x.c + y.c}; }
__host__ __device__ __forceinline__ V3 v3_sub(V3 x, V3 y) { return V3{x.a - y.a, x.b - y.b, x.c - y.c}; }
// x + M y, M's element i at m[i * ST]
template <int ST>
__host__ __device__ __forceinline__ V3 mv_add(V3 x, const double *m, V3 y) {
    return V3{fma(m[0], y.a, fma(m[ST], y.b, fma(m[2 * ST], y.c, x.a))),
              fma(m[3 * ST], y.a, fma(m[4 * ST], y.b, fma(m[5 * ST], y.c, x.b))),
              fma(m[6 * ST], y.a, fma(m[7 * ST], y.b, fma(m[8 * ST], y.c, x.c)))};
}

struct Beta {
    double b1, b2, b3;
};
// The filter's next value from its input and its last three, and the last three after it.
__host__ __device__ __forceinline__ double filter(const Beta &be, double in, const V3 &s) {
    return fma(-be.b1, s.a, fma(-be.b2, s.b, fma(-be.b3, s.c, in)));
}
__host__ __device__ __forceinline__ V3 shift(double x, const V3 &s) { return V3{x, s.a, s.b}; }

// H z (H is symmetric; rows past the last of a call's, if it has fewer than
// three, see zeta = 0 and change nothing).
__host__ __device__ __forceinline__ V3 hankel(const Beta &be, V3 z) {
    return V3{fma(be.b1, z.a, fma(be.b2, z.b, be.b3 * z.c)), fma(be.b2, z.a, be.b3 * z.b), be.b3 * z.a};
}

// G and the head response R of n rows, by recursion.
__host__ __device__ inline void row_responses(int n, const Beta &be, double (&R)[9], double (&G)[9]) {
    V3 h{0.0, 0.0, 0.0}, v[3] = {{1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {0.0, 0.0, 1.0}};
    double in = 1.0, g[6] = {};
#pragma unroll
    for (int i = 0; i < 9; ++i) R[i] = 0.0;
    for (int k = 0; k < n; ++k) {
        h = shift(filter(be, in, h), h);
        in = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            v[c] = shift(filter(be, 0.0, v[c]), v[c]);
            R[c] = fma(v[c].a, h.a, R[c]);
            R[3 + c] = fma(v[c].a, h.b, R[3 + c]);
            R[6 + c] = fma(v[c].a, h.c, R[6 + c]);
        }
        g[0] = fma(h.a, h.a, g[0]);
        g[1] = fma(h.a, h.b, g[1]);
        g[2] = fma(h.a, h.c, g[2]);
        g[3] = fma(h.b, h.b, g[3]);
        g[4] = fma(h.b, h.c, g[4]);
        g[5] = fma(h.c, h.c, g[5]);
    }
    const double s[9] = {g[0], g[1], g[2], g[1], g[3], g[4], g[2], g[4], g[5]};
#pragma unroll
    for (int i = 0; i < 9; ++i) G[i] = s[i];
}

// S = I + H G H as its Cholesky factor, the diagonal as reciprocals.  S has no
// eigenvalue below 1, so no pivot is below 1 but by rounding.
struct Corner {
    double i0, l10, l20, i1, l21, i2;
};
__host__ __device__ inline Corner corner(const Beta &be, const double (&G)[9]) {
    const double H[9] = {be.b1, be.b2, be.b3, be.b2, be.b3, 0.0, be.b3, 0.0, 0.0};
    double t[9], S[9];
    mat_mul(t, G, H);
    mat_mul(S, H, t);
    Corner c;
    c.i0 = 1.0 / sqrt(1.0 + S[0]);
    c.l10 = S[3] * c.i0;
    c.l20 = S[6] * c.i0;
    c.i1 = 1.0 / sqrt(fmax(1.0, fma(-c.l10, c.l10, 1.0 + S[4])));
    c.l21 = fma(-c.l20, c.l10, S[7]) * c.i1;
    c.i2 = 1.0 / sqrt(fmax(1.0, fma(-c.l21, c.l21, fma(-c.l20, c.l20, 1.0 + S[8]))));
    return c;
}
// What the solve loses in a branch: the trace of G over the plan's rows, which is how
// far the filters carry rounding, times the second pivot of S, which is how much of
// it the corner's equations for t (nearly dependent where zeros are together near
// the circle) let through.  Over 1200 sets of taps (double and triple zeros at
// moduli 0.9 to 1, mirrored or not; Gaussian, Kaiser, Hamming-like, triangular and
// sinc windows) and 20 to 4096 rows, up to LOSS_MAX the solve is at most 1.1e-8 of a
// branch's rms off, so at most 7% above the FP32 rounding of the output (2.8e-8) or
// the factor rows' error; the first case that is neither below 1.5e-8 nor below the
// factor rows' lies at 1.7 times LOSS_MAX, a window of three zeros near -1 (a
// Gaussian of sigma 0.954 blocks) at thousands of times.  Hann-sinc has 7e2, the Hamming
// prototype 5.8e8: at 4096 rows the solve loses up to 4e-9 there, the factor rows 5e-7.
constexpr double LOSS_MAX = 1e9;
__host__ __device__ __forceinline__ bool admitted(double loss) { return loss <= LOSS_MAX; }   // NaN: not

// The tables of one branch (row k at tab[k * stride]) for plans of up to `blocks`
// blocks; returns what the solve loses in it.  The block's responses come by recursion over their rows in
// double-double, so that the tables' rounding is that of their last digit (powers by
// squaring in FP64 lose 3e-7 of the result on the Hamming prototype).
__host__ __device__ inline double plan_tables(const float (&taps)[4], int blocks, double *tab, size_t stride) {
    const double w[4] = {taps[0], taps[1], taps[2], taps[3]};
    Dd b[4];
    min_phase(w, b);
    const double be1 = dd_div(b[1], b[0]).h, be2 = dd_div(b[2], b[0]).h, be3 = dd_div(b[3], b[0]).h;
    tab[(TB_BETA + 0) * stride] = be1;
    tab[(TB_BETA + 1) * stride] = be2;
    tab[(TB_BETA + 2) * stride] = be3;
    const Dd bb = dd_mul(b[0], b[0]);
    for (int i = 0; i < 4; ++i) tab[(TB_WZ + i) * stride] = dd_div(dd(w[i]), bb).h;
    Dd v[3][3] = {{{1.0, 0.0}, {}, {}}, {{}, {1.0, 0.0}, {}}, {{}, {}, {1.0, 0.0}}};   // chain c: its last three values
    Dd h[3] = {}, rm[9] = {}, g[6] = {};
    const Dd n1 = dd(be1), n2 = dd(be2), n3 = dd(be3);
    double CB[9];
    for (int k = 0; k < SBLK; ++k) {
        const Dd hk = dd_sub_mul(dd_sub_mul(dd_sub_mul(dd(k == 0 ? 1.0 : 0.0), h[0], n1), h[1], n2), h[2], n3);
        h[2] = h[1];
        h[1] = h[0];
        h[0] = hk;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const Dd x = dd_sub_mul(dd_sub_mul(dd_sub_mul(Dd{}, v[c][0], n1), v[c][1], n2), v[c][2], n3);
            v[c][2] = v[c][1];
            v[c][1] = v[c][0];
            v[c][0] = x;
#pragma unroll
            for (int r = 0; r < 3; ++r) rm[3 * r + c] = dd_add(rm[3 * r + c], dd_mul(x, h[r]));
        }
#pragma unroll
        for (int r = 0, i = 0; r < 3; ++r)
#pragma unroll
            for (int c = r; c < 3; ++c, ++i) g[i] = dd_add(g[i], dd_mul(h[r], h[c]));
        if (k >= SBLK - 5) tab[(TB_HB + k - (SBLK - 5)) * stride] = hk.h;
        if (k == SR - 1 || k == SBLK - 1) {
            const int row = k == SR - 1 ? TB_CS : TB_CB;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) tab[(row + 3 * r + c) * stride] = CB[3 * r + c] = v[c][r].h;
        }
    }
    for (int i = 0; i < 9; ++i) tab[(TB_RB + i) * stride] = rm[i].h;
    const double GB[9] = {g[0].h, g[1].h, g[2].h, g[1].h, g[3].h, g[4].h, g[2].h, g[4].h, g[5].h};
    for (int i = 0; i < 9; ++i) tab[(TB_GB + i) * stride] = GB[i];
    double P[9], G[9];
    block_gram(blocks, CB, GB, P, G);
    // of the plan's rows and of one block, whose G has no rounding of powers in it
    const Corner c = corner(Beta{be1, be2, be3}, G), c1 = corner(Beta{be1, be2, be3}, GB);
    const double loss = (G[0] + G[4] + G[8]) / (c.i1 * c.i1), loss1 = (GB[0] + GB[4] + GB[8]) / (c1.i1 * c1.i1);
    return loss1 <= LOSS_MAX && !(loss < loss1) ? loss : loss1;      // NaN stays
}

// One step of t: what it changes by, with zeta the head of the solution that t gives.
__host__ __device__ __forceinline__ V3 corner_step(const Corner &c, const Beta &be, V3 zeta, V3 t) {
    const V3 r = v3_sub(hankel(be, zeta), t);
    const double y0 = r.a * c.i0, y1 = (r.b - c.l10 * y0) * c.i1, y2 = (r.c - c.l20 * y0 - c.l21 * y1) * c.i2;
    const double z2 = y2 * c.i2, z1 = (y1 - c.l21 * z2) * c.i1;
    return V3{(y0 - c.l10 * z1 - c.l20 * z2) * c.i0, z1, z2};
}
// Steps of t: from nothing and one of refinement wherever it is sought; the
// block that holds the corner takes one more from its own rows, since t rounded
// as it comes from the join is (B B^T)^-1's first columns off.
constexpr int CORNER_STEPS = 2, CORNER_STEPS_BLOCK = 1;

}  // namespace pfb
}  // namespace sdbe
