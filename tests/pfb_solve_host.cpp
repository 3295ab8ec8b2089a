// Host build of the PFB inverse's constant-coefficient solve
// (sdbe_amd/csrc/sdbe_pfb_solve.hpp), one branch at a time, for
// test_pfb_solve_host.py: the functions the kernels call, put together in the order
// of k_pfb_span, k_pfb_join and k_pfb_solve (blocks of 256 rows, spans of 32), beside
// the banded Cholesky solve of P P^T in 80-bit and in FP64 arithmetic.
#define __host__
#define __device__
#define __forceinline__ inline
#include "../sdbe_amd/csrc/sdbe_pfb_solve.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

using namespace sdbe::pfb;

namespace {

using Vec = std::vector<double>;

template <typename T>
Vec cholesky(const float *w, const std::vector<float> &y) {
    const int N = (int)y.size();
    T a[4];
    for (int d = 0; d < 4; ++d) {
        a[d] = 0;
        for (int k = 0; k + d < 4; ++k) a[d] += (T)w[k + d] * (T)w[k];
    }
    std::vector<T> L(4 * (size_t)N), z(N);         // L(i, i - d) at 4 i + d
    for (int i = 0; i < N; ++i) {
        T r = y[i];
        for (int d = std::min(i, 3); d >= 0; --d) {
            const int j = i - d;
            T s = a[d];
            for (int k = std::max(i - 3, 0); k < j; ++k)
                if (j - k <= 3) s -= L[4 * i + i - k] * L[4 * j + j - k];
            L[4 * i + d] = d ? s / L[4 * j] : std::sqrt(s);
            if (d) r -= L[4 * i + d] * z[j];
        }
        z[i] = r / L[4 * i];
    }
    for (int i = N - 1; i >= 0; --i) {
        T r = z[i];
        for (int d = 1; d < 4 && i + d < N; ++d) r -= L[4 * (i + d) + d] * z[i + d];
        z[i] = r / L[4 * i];
    }
    Vec x(N + 3);
    for (int i = 0; i < N + 3; ++i) {
        T s = 0;
        for (int k = 0; k < 4; ++k)
            if (i - k >= 0 && i - k < N) s += (T)w[k] * z[i - k];
        x[i] = (double)s;
    }
    return x;
}

const V3 ZERO{0.0, 0.0, 0.0};
V3 neg(V3 a) { return V3{-a.a, -a.b, -a.c}; }

struct Branch {
    double tab[TB_N];
    Beta be;
    double loss;
    Branch(const float *w, int blocks) {
        const float t[4] = {w[0], w[1], w[2], w[3]};
        loss = plan_tables(t, blocks, tab, 1);
        be = Beta{tab[0], tab[1], tab[2]};
    }
};

// k_pfb_solve
void block(const Branch &br, const std::vector<float> &y, int blk, bool one, const Corner &cn, V3 tt, V3 c0, V3 b0,
           Vec &x) {
    const int N = (int)y.size();
    const double *cs = br.tab + TB_CS, *W = br.tab + TB_WZ;
    const Beta &be = br.be;
    double v[SWV][SR];
    V3 tot[SWV], q[SWV], b[SWV];
    auto rows = [&](int w) { return N - (SBLK * blk + SR * w); };
    auto change = [&](int w, V3 in, V3 d) {
        for (int k = 0; k < SR; ++k) {
            const double dk = filter(be, k == 0 ? -in.a : k == 1 ? -in.b : k == 2 ? -in.c : 0.0, d);
            v[w][k] = k < rows(w) ? v[w][k] + dk : 0.0;
            d = shift(dk, d);
        }
        return d;
    };
    const V3 g = hankel(be, tt);
    for (int w = 0; w < SWV; ++w) {
        V3 p = ZERO;
        for (int k = 0; k < SR; ++k) {
            double in = k < rows(w) ? y[SBLK * blk + SR * w + k] : 0.0;
            if (w == 0 && k < 3) in -= k == 0 ? g.a : k == 1 ? g.b : g.c;
            v[w][k] = filter(be, in, p);
            p = shift(v[w][k], p);
        }
        tot[w] = p;
    }
    for (int w = 0; w < SWV; ++w) {
        V3 a = c0;
        for (int i = 0; i < w; ++i) a = mv_add<1>(tot[i], cs, a);
        change(w, ZERO, a);
    }
    const int steps = one ? CORNER_STEPS : blk == 0 ? CORNER_STEPS_BLOCK : 0;
    for (int it = 0;; ++it) {
        for (int w = 0; w < SWV; ++w) {
            q[w] = ZERO;
            for (int k = SR - 1; k >= 0; --k) q[w] = shift(filter(be, v[w][k], q[w]), q[w]);
        }
        for (int w = 0; w < SWV; ++w) {
            b[w] = b0;
            for (int i = SWV - 1; i > w; --i) b[w] = mv_add<1>(q[i], cs, b[w]);
        }
        if (it == steps) break;
        const V3 dt = corner_step(cn, be, mv_add<1>(q[0], cs, b[0]), tt);
        tt = v3_add(tt, dt);
        V3 d = change(0, hankel(be, dt), ZERO);
        for (int w = 1; w < SWV; ++w) {
            change(w, ZERO, d);
            d = mv_add<1>(ZERO, cs, d);
        }
    }
    for (int w = 0; w < SWV && rows(w) > 0; ++w) {
        V3 s = b[w];
        const int r0 = SBLK * blk + SR * w;
        for (int k = SR - 1; k >= 0; --k) {
            const double z = filter(be, v[w][k], s);
            if (k < rows(w)) x[r0 + k + 3] = W[0] * s.c + W[1] * s.b + W[2] * s.a + W[3] * z;
            s = shift(z, s);
        }
        if (r0 == 0) {
            x[2] = W[0] * s.c + W[1] * s.b + W[2] * s.a;
            x[1] = W[0] * s.b + W[1] * s.a;
            x[0] = W[0] * s.a;
        }
    }
}

Vec constant_solve(const Branch &br, const std::vector<float> &y) {
    const int N = (int)y.size(), nb = (N + SBLK - 1) / SBLK, last = (N - 1) % SBLK + 1;
    const Beta &be = br.be;
    Vec x(N + 3);
    double R[9], G[9];
    if (nb == 1) {
        row_responses(N, be, R, G);
        block(br, y, 0, true, corner(be, G), ZERO, ZERO, ZERO, x);
        return x;
    }
    std::vector<V3> P(nb), Q(nb), A(nb), B(nb), q(nb);
    for (int k = 0; k < nb; ++k) {                    // k_pfb_span
        V3 st = ZERO, h = ZERO, s = ZERO;
        for (int i = SBLK * k; i < std::min(SBLK * (k + 1), N); ++i) {
            st = shift(filter(be, y[i], st), st);
            h = shift(filter(be, i == SBLK * k ? 1.0 : 0.0, h), h);
            s = V3{std::fma(st.a, h.a, s.a), std::fma(st.a, h.b, s.b), std::fma(st.a, h.c, s.c)};
        }
        P[k] = st;
        Q[k] = s;
    }
    double cb[9], rb[9], gb[9], rl[9], pw[9];         // k_pfb_join
    for (int i = 0; i < 9; ++i) {
        cb[i] = br.tab[TB_CB + i];
        rl[i] = rb[i] = br.tab[TB_RB + i];
        gb[i] = br.tab[TB_GB + i];
    }
    block_gram(last == SBLK ? nb : nb - 1, cb, gb, pw, G);
    if (last != SBLK) {
        double gl[9], s[9], u[9];
        row_responses(last, be, rl, gl);
        mat_mul(s, pw, gl);
        mat_mul_t(u, s, pw);
        for (int i = 0; i < 9; ++i) G[i] += u[i];
    }
    const Corner cn = corner(be, G);
    const double *h = br.tab + TB_HB;
    V3 tt = ZERO;
    for (int it = 0;; ++it) {
        const V3 g = hankel(be, tt);
        V3 a = ZERO, z = ZERO;
        for (int k = 0; k < nb; ++k) {
            V3 p = P[k], s = Q[k];
            if (k == 0) {
                p = v3_sub(p, V3{g.a * h[4] + g.b * h[3] + g.c * h[2], g.a * h[3] + g.b * h[2] + g.c * h[1],
                                 g.a * h[2] + g.b * h[1] + g.c * h[0]});
                s = mv_add<1>(s, gb, neg(g));
            }
            A[k] = a;
            q[k] = mv_add<1>(s, k == nb - 1 ? rl : rb, a);
            a = mv_add<1>(p, cb, a);
        }
        for (int k = nb - 1; k >= 0; --k) {
            B[k] = z;
            z = mv_add<1>(q[k], cb, z);
        }
        if (it == CORNER_STEPS) break;
        tt = v3_add(tt, corner_step(cn, be, z, tt));
    }
    for (int k = 0; k < nb; ++k) block(br, y, k, false, cn, k == 0 ? tt : ZERO, A[k], B[k], x);
    return x;
}

double rel(const Vec &a, const Vec &b) {
    double e = 0.0, s = 0.0;
    for (size_t i = 0; i < a.size(); ++i) {
        e += (a[i] - b[i]) * (a[i] - b[i]);
        s += b[i] * b[i];
    }
    return std::sqrt(e / s);
}

}  // namespace

extern "C" {

// Which of n branches (taps [n][4]) plans of up to `blocks` blocks admit.
void admit(int n, const float *taps, int blocks, int *out) {
    for (int i = 0; i < n; ++i) out[i] = admitted(Branch(taps + 4 * (size_t)i, blocks).loss);
}

// Largest difference of the factor's autocorrelation from the taps', of their lag 0.
double factor_error(const float *taps) {
    const double w[4] = {taps[0], taps[1], taps[2], taps[3]};
    Dd b[4];
    min_phase(w, b);
    long double worst = 0, a0 = 0;
    for (int d = 0; d < 4; ++d) {
        long double p = 0, q = 0;
        for (int k = 0; k + d < 4; ++k) {
            p += (long double)w[k] * w[k + d];
            q += ((long double)b[k].h + b[k].l) * ((long double)b[k + d].h + b[k + d].l);
        }
        if (d == 0) a0 = p;
        worst = std::max(worst, std::fabs(p - q));
    }
    return (double)(worst / a0);
}

// Relative rms errors of the constant-coefficient solve and of the FP64 factor
// rows against 80 bits, for the right-hand side y of N rows.
void errors(const float *taps, int N, const float *y, int blocks, double *out) {
    const std::vector<float> v(y, y + N);
    const Vec want = cholesky<long double>(taps, v);
    out[0] = rel(constant_solve(Branch(taps, blocks), v), want);
    out[1] = rel(cholesky<double>(taps, v), want);
}
}
