// Polynomial roots of the shape tests (gfx950), in the reference's operation
// order.  Plain arithmetic only, so the same source also builds for the host
// (the CPU tests compare it with the oracle's solver).
#ifndef PVX_POLY_DEVICE_H
#define PVX_POLY_DEVICE_H

#include <math.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define PVX_POLY_FN __device__ inline
#else
#define PVX_POLY_FN inline
#endif

#include "pvx_types.h"

namespace pvx {

// ---------------------------------------------------------------------------
// Polynomial roots: core/math/polynomialsolver.cpp (default build branches).
// sbisect's recursion becomes an explicit interval stack visited
// left-to-right, which yields the same roots in the same order.
// ---------------------------------------------------------------------------
namespace poly {
constexpr int kMaxIter = 50;
constexpr double kSmall = 1.0e-10;
constexpr double kRel = 1.0e-12;

// A polynomial of order <= N, ascending powers (the reference's `polynomial`
// holds up to MAX_ORDER 35; the shapes here need 4 (torus) and 6 (lathe)).
template <int N>
struct PN {
    int ord;
    double c[N + 1];
};
using P4 = PN<4>;

PVX_POLY_FN double eval(double x, int n, const double *c) {
    double v = c[n];
    for (int i = n - 1; i >= 0; i--) v = v * x + c[i];
    return v;
}

template <int N>
PVX_POLY_FN int modp(const PN<N> &u, const PN<N> &v, PN<N> &r) {
    r = u;
    if (v.c[v.ord] < 0.0) {
        for (int k = u.ord - v.ord - 1; k >= 0; k -= 2) r.c[k] = -r.c[k];
        for (int k = u.ord - v.ord; k >= 0; k--)
            for (int j = v.ord + k - 1; j >= k; j--) r.c[j] = -r.c[j] - r.c[v.ord + k] * v.c[j - k];
    } else {
        for (int k = u.ord - v.ord; k >= 0; k--)
            for (int j = v.ord + k - 1; j >= k; j--) r.c[j] -= r.c[v.ord + k] * v.c[j - k];
    }
    int k = v.ord - 1;
    while (k >= 0 && fabs(r.c[k]) < kSmall) {
        r.c[k] = 0.0;
        k--;
    }
    r.ord = (k < 0) ? 0 : k;
    return r.ord;
}

template <int N>
PVX_POLY_FN int buildsturm(int ord, PN<N> *s) {
    s[0].ord = ord;
    s[1].ord = ord - 1;
    double f = fabs(s[0].c[ord] * ord);
    for (int i = 1; i <= ord; i++) s[1].c[i - 1] = s[0].c[i] * i / f;
    int k = 2;
    while (modp(s[k - 2], s[k - 1], s[k])) {
        f = -fabs(s[k].c[s[k].ord]);
        for (int j = s[k].ord; j >= 0; j--) s[k].c[j] /= f;
        k++;
    }
    s[k].c[0] = -s[k].c[0];
    return k;
}

template <int N>
PVX_POLY_FN int numchanges(int np, const PN<N> *s, double a) {
    int ch = 0;
    double lf = eval(a, s[0].ord, s[0].c);
    for (int k = 1; k <= np; k++) {
        double f = eval(a, s[k].ord, s[k].c);
        if (lf == 0.0 || lf * f < 0) ch++;
        lf = f;
    }
    return ch;
}

template <int N>
PVX_POLY_FN int visible_roots(int np, const PN<N> *s) {
    int atpos = 0, atzero = 0;
    double lf = s[0].c[s[0].ord];
    for (int k = 1; k <= np; k++) {
        double f = s[k].c[s[k].ord];
        if (lf == 0.0 || lf * f < 0) atpos++;
        lf = f;
    }
    lf = s[0].c[0];
    for (int k = 1; k <= np; k++) {
        double f = s[k].c[0];
        if (lf == 0.0 || lf * f < 0) atzero++;
        lf = f;
    }
    return atzero - atpos;
}

PVX_POLY_FN int regula_falsa(int order, const double *coef, double a, double b, double *val) {
    double fa = eval(a, order, coef), fb = eval(b, order, coef), x, fx, lfx;
    if (fa * fb > 0.0) return 0;
    if (fabs(fa) < kSmall) { *val = a; return 1; }
    if (fabs(fb) < kSmall) { *val = b; return 1; }
    lfx = fa;
    for (int its = 0; its < kMaxIter; its++) {
        x = (fb * a - fa * b) / (fb - fa);
        fx = eval(x, order, coef);
        if (fabs(x) > kRel) {
            if (fabs(fx / x) < kRel) { *val = x; return 1; }
        } else if (fabs(fx) < kRel) {
            *val = x;
            return 1;
        }
        if (fa < 0) {
            if (fx < 0) { a = x; fa = fx; if ((lfx * fx) > 0) fb /= 2; }
            else { b = x; fb = fx; if ((lfx * fx) > 0) fa /= 2; }
        } else {
            if (fx < 0) { b = x; fb = fx; if ((lfx * fx) > 0) fa /= 2; }
            else { a = x; fa = fx; if ((lfx * fx) > 0) fb /= 2; }
        }
        if (fabs(b - a) < kRel) { *val = x; return 1; }
        lfx = fx;
    }
    return 0;
}

// sbisect over an explicit stack.
template <int N>
PVX_POLY_FN int sbisect(int np, const PN<N> *s, double lo, double hi, int atlo, int athi,
                              double *roots) {
    struct Iv {
        double lo, hi;
        int atlo, athi;
    } st[N + 2]; // each pending interval holds at least one of the <= N roots
    int sp = 0, nr = 0;
    st[sp++] = Iv{lo, hi, atlo, athi};
    while (sp > 0) {
        Iv iv = st[--sp];
        double mn = iv.lo, mx = iv.hi, mid = 0.0;
        int amin = iv.atlo, amax = iv.athi;
        if (amin - amax == 1) {
            if (regula_falsa(s[0].ord, s[0].c, mn, mx, &roots[nr])) {
                nr++;
                continue;
            }
            bool done = false;
            for (int its = 0; its < kMaxIter; its++) {
                mid = (mn + mx) / 2;
                int am = numchanges(np, s, mid);
                if (am < amax || am > amin) { done = true; break; } // no root
                if (fabs(mid) > kRel) {
                    if (fabs((mx - mn) / mid) < kRel) { roots[nr++] = mid; done = true; break; }
                } else if (fabs(mx - mn) < kRel) {
                    roots[nr++] = mid;
                    done = true;
                    break;
                }
                if (amin - am == 0) mn = mid; else mx = mid;
            }
            if (!done) roots[nr++] = mid;
            continue;
        }
        bool handled = false;
        for (int its = 0; its < kMaxIter; its++) {
            mid = (mn + mx) / 2;
            int am = numchanges(np, s, mid);
            if (am < amax || am > amin) { handled = true; break; }
            if (fabs(mid) > kRel) {
                if (fabs((mx - mn) / mid) < kRel) { roots[nr++] = mid; handled = true; break; }
            } else if (fabs(mx - mn) < kRel) {
                roots[nr++] = mid;
                handled = true;
                break;
            }
            int n1 = amin - am, n2 = am - amax;
            if (n1 != 0 && n2 != 0) {
                if (sp + 2 <= N + 2) {
                    st[sp++] = Iv{mid, mx, am, amax}; // right, visited second
                    st[sp++] = Iv{mn, mid, amin, am}; // left, visited first
                }
                handled = true;
                break;
            }
            if (n1 == 0) mn = mid; else mx = mid;
        }
        if (!handled) roots[nr++] = mid;
    }
    return nr;
}

// (an order-N polynomial has at most N roots pending on the interval stack)
template <int N = 4>
PVX_POLY_FN int polysolve(int order, const double *coeffs, double *roots) {
    PN<N> s[N + 2];
    for (int i = 0; i <= order; i++) s[0].c[order - i] = coeffs[i] / coeffs[0];
    int np = buildsturm(order, s);
    if (visible_roots(np, s) == 0) return 0;
    int atmin = numchanges(np, s, 0.0);
    int atmax = numchanges(np, s, kMaxDistance);
    if (atmin - atmax == 0) return 0;
    return sbisect(np, s, 0.0, kMaxDistance, atmin, atmax, roots);
}

// ---------------------------------------------------------------------------
// The same Sturm solver with the whole chain in registers, for a polynomial
// of exactly order N whose remainders drop one degree each (all but
// degenerate ones): every index is static, so nothing lives in the per-lane
// stack.  Same operations in the same order as polysolve, hence the same
// roots bit for bit.  What bound the stack form was its loads: one torus
// takes some hundred Horner steps on the chain, each a dependent private
// memory access.
// ---------------------------------------------------------------------------
// fabs(a / b) < kRel for fabs(b) > kRel; the division itself is made only
// when the quotient is within 1e-14 of the limit.
PVX_POLY_FN bool ratio_small(double a, double b) {
    const double x = fabs(a), y = kRel * fabs(b);
    if (x < y * (1.0 - 1.0e-14)) return true;
    if (x > y * (1.0 + 1.0e-14)) return false;
    return fabs(a / b) < kRel;
}

template <int N>
struct Chain {
    double c[N + 1][N + 1]; // c[k]: degree N - k, ascending powers

    template <int K>
    PVX_POLY_FN double at(double x) const {
        double v = c[K][N - K];
#pragma unroll
        for (int i = N - K - 1; i >= 0; i--) v = v * x + c[K][i];
        return v;
    }
    template <int K>
    PVX_POLY_FN int changes_from(double x, double lf) const {
        if constexpr (K > N) {
            return 0;
        } else {
            const double f = at<K>(x);
            return ((lf == 0.0 || lf * f < 0) ? 1 : 0) + changes_from<K + 1>(x, f);
        }
    }
    PVX_POLY_FN int numchanges(double x) const { return changes_from<1>(x, at<0>(x)); }
    // remainder K of the sequence; false: it drops more than one degree
    template <int K>
    PVX_POLY_FN bool build_from() {
        if constexpr (K > N) {
            return true;
        } else {
            constexpr int du = N - K + 2, dv = N - K + 1; // degrees of c[K-2], c[K-1]
            const bool neg = c[K - 1][dv] < 0.0;
            double r[du + 1];
#pragma unroll
            for (int j = 0; j <= du; j++) r[j] = c[K - 2][j];
            if (neg) r[0] = -r[0];
#pragma unroll
            for (int k = 1; k >= 0; k--)
#pragma unroll
                for (int j = dv + k - 1; j >= k; j--) r[j] = (neg ? -r[j] : r[j]) - r[dv + k] * c[K - 1][j - k];
            if constexpr (dv - 1 > 0) {
                if (fabs(r[dv - 1]) < kSmall) return false;
                const double f = -fabs(r[dv - 1]);
#pragma unroll
                for (int j = dv - 1; j >= 0; j--) c[K][j] = r[j] / f;
            } else {
                if (fabs(r[0]) < kSmall) r[0] = 0.0;
                c[K][0] = -r[0];
            }
            return build_from<K + 1>();
        }
    }
    // leading coefficients' sign changes (at infinity)
    template <int K>
    PVX_POLY_FN int lead_changes(double lf) const {
        if constexpr (K > N) {
            return 0;
        } else {
            const double f = c[K][N - K];
            return ((lf == 0.0 || lf * f < 0) ? 1 : 0) + lead_changes<K + 1>(f);
        }
    }
    template <int K>
    PVX_POLY_FN int zero_changes(double lf) const {
        if constexpr (K > N) {
            return 0;
        } else {
            const double f = c[K][0];
            return ((lf == 0.0 || lf * f < 0) ? 1 : 0) + zero_changes<K + 1>(f);
        }
    }
    // Beyond this every c[k] has its leading coefficient's sign, also as
    // evaluated: with the other coefficients' magnitudes summing to M and a
    // leading one of magnitude 1, each Horner step at x >= 2 + 2 M keeps that
    // sign and grows.  (NaN when a coefficient is: no x is beyond it.)
    PVX_POLY_FN double beyond() const {
        double m = 0.0;
        bool unit = true;
#pragma unroll
        for (int k = 0; k < N; k++) {
            unit = unit && fabs(c[k][N - k]) == 1.0;
#pragma unroll
            for (int i = 0; i < N - k; i++) m += fabs(c[k][i]);
        }
        return unit ? 2.0 + 2.0 * m : HUGE_VAL;
    }
    // regula_falsa on c[0]
    PVX_POLY_FN bool regula(double a, double b, double &val) const {
        double fa = at<0>(a), fb = at<0>(b), x, fx, lfx;
        if (fa * fb > 0.0) return false;
        if (fabs(fa) < kSmall) { val = a; return true; }
        if (fabs(fb) < kSmall) { val = b; return true; }
        lfx = fa;
        for (int its = 0; its < kMaxIter; its++) {
            x = (fb * a - fa * b) / (fb - fa);
            fx = at<0>(x);
            if (fabs(x) > kRel) {
                if (ratio_small(fx, x)) { val = x; return true; }
            } else if (fabs(fx) < kRel) {
                val = x;
                return true;
            }
            const bool half = lfx * fx > 0;
            if ((fa < 0) == (fx < 0)) { // the low end moves
                a = x;
                fa = fx;
                if (half) fb /= 2;
            } else {
                b = x;
                fb = fx;
                if (half) fa /= 2;
            }
            if (fabs(b - a) < kRel) { val = x; return true; }
            lfx = fx;
        }
        return false;
    }
};

// Stores root number n (static indices only).
template <int N>
PVX_POLY_FN void put_root(double (&r)[N], int &n, double v) {
#pragma unroll
    for (int j = 0; j < N; j++)
        if (n == j) r[j] = v;
    n++;
}

// polysolve of order N on `coeffs` (descending); -1: a degenerate chain, to
// be solved by polysolve.
template <int N>
PVX_POLY_FN int polysolve_reg(const double *coeffs, double (&roots)[N]) {
    Chain<N> s;
#pragma unroll
    for (int i = 0; i <= N; i++) s.c[0][N - i] = coeffs[i];
    if (coeffs[0] != 1.0)
#pragma unroll
        for (int i = 0; i <= N; i++) s.c[0][i] /= coeffs[0];
    {
        const double f = fabs(s.c[0][N] * N);
        if (f == 4.0) { // a power of two: the product is the quotient
#pragma unroll
            for (int i = 1; i <= N; i++) s.c[1][i - 1] = s.c[0][i] * i * 0.25;
        } else {
#pragma unroll
            for (int i = 1; i <= N; i++) s.c[1][i - 1] = s.c[0][i] * i / f;
        }
    }
    if (!s.template build_from<2>()) return -1;
    const int lead = s.template lead_changes<1>(s.c[0][N]);
    if (s.template zero_changes<1>(s.c[0][0]) - lead == 0) return 0;
    // sign changes at x: known without evaluation beyond every polynomial's
    // roots, which two thirds of the halvings of [0, kMaxDistance] are
    const double far = s.beyond();
    auto changes = [&](double x) { return x >= far ? lead : s.numchanges(x); };
    int amin = s.numchanges(0.0), amax = changes(kMaxDistance);
    if (amin - amax == 0) return 0;
    // sbisect: the interval at hand, and the ones to its right that wait
    // (each holds a root, so at most N - 1 wait)
    double mn = 0.0, mx = kMaxDistance, plo[N - 1], phi[N - 1];
    int pmin[N - 1], pmax[N - 1], sp = 0, nr = 0;
    for (;;) {
        double mid = 0.0;
        bool split = false;
        if (amin - amax == 1) {
            double v;
            if (s.regula(mn, mx, v)) {
                put_root(roots, nr, v);
            } else {
                bool root = true;
                for (int its = 0; its < kMaxIter; its++) {
                    mid = (mn + mx) / 2;
                    const int am = changes(mid);
                    if (am < amax || am > amin) { root = false; break; }
                    if (fabs(mid) > kRel) {
                        if (ratio_small(mx - mn, mid)) break;
                    } else if (fabs(mx - mn) < kRel) {
                        break;
                    }
                    if (amin - am == 0) mn = mid; else mx = mid;
                }
                if (root) put_root(roots, nr, mid);
            }
        } else {
            bool root = true;
            for (int its = 0; its < kMaxIter; its++) {
                mid = (mn + mx) / 2;
                const int am = changes(mid);
                if (am < amax || am > amin) { root = false; break; }
                if (fabs(mid) > kRel) {
                    if (ratio_small(mx - mn, mid)) break;
                } else if (fabs(mx - mn) < kRel) {
                    break;
                }
                const int n1 = amin - am, n2 = am - amax;
                if (n1 != 0 && n2 != 0) { // the right half waits, the left one is next
#pragma unroll
                    for (int j = 0; j < N - 1; j++)
                        if (sp == j) {
                            plo[j] = mid;
                            phi[j] = mx;
                            pmin[j] = am;
                            pmax[j] = amax;
                        }
                    sp++;
                    mx = mid;
                    amax = am;
                    split = true;
                    break;
                }
                if (n1 == 0) mn = mid; else mx = mid;
            }
            if (root && !split) put_root(roots, nr, mid);
        }
        if (split) continue;
        if (sp == 0) break;
        sp--;
#pragma unroll
        for (int j = 0; j < N - 1; j++)
            if (sp == j) {
                mn = plo[j];
                mx = phi[j];
                amin = pmin[j];
                amax = pmax[j];
            }
    }
    return nr;
}

// polysolve of order 3 or 4 into four root places.
template <int N>
PVX_POLY_FN int polysolve_n(const double *c, double *r) {
    double v[N];
    const int n = polysolve_reg<N>(c, v);
    if (n < 0) return polysolve<N>(N, c, r);
#pragma unroll
    for (int j = 0; j < N; j++)
        if (j < n) r[j] = v[j];
    return n;
}

PVX_POLY_FN int solve_quadratic(const double *x, double *y) {
    double a = x[0], b = -x[1], c = x[2];
    if (a == 0.0) {
        if (b == 0.0) return 0;
        y[0] = c / b;
        return 1;
    }
    b /= a;
    c /= a;
    a = 1.0;
    double d = b * b - 4.0 * a * c;
    if (d > -kSmall && d < kSmall) {
        y[0] = 0.5 * b / a;
        return 1;
    }
    if (d < 0.0) return 0;
    d = sqrt(d);
    double t = 2.0 * a;
    y[0] = (b + d) / t;
    y[1] = (b - d) / t;
    return 2;
}

PVX_POLY_FN int solve_cubic(const double *x, double *y) {
    double a0 = x[0], a1, a2, a3;
    if (a0 == 0.0) return solve_quadratic(&x[1], y);
    if (a0 != 1.0) {
        a1 = x[1] / a0; a2 = x[2] / a0; a3 = x[3] / a0;
    } else {
        a1 = x[1]; a2 = x[2]; a3 = x[3];
    }
    double A2 = a1 * a1;
    double Q = (A2 - 3.0 * a2) / 9.0;
    double R = (a1 * (A2 - 4.5 * a2) + 13.5 * a3) / 27.0;
    double Q3 = Q * Q * Q, R2 = R * R, dd = Q3 - R2, an = a1 / 3.0;
    if (dd >= 0.0) {
        dd = R / sqrt(Q3);
        double theta = acos(dd) / 3.0;
        double sQ = -2.0 * sqrt(Q);
        y[0] = sQ * cos(theta) - an;
        y[1] = sQ * cos(theta + 2.0943951023931954923084) - an;
        y[2] = sQ * cos(theta + 4.1887902047863909846168) - an;
        return 3;
    }
    double sQ = pow(sqrt(R2 - Q3) + fabs(R), 1.0 / 3.0);
    y[0] = (R < 0) ? (sQ + Q / sQ) - an : -(sQ + Q / sQ) - an;
    return 1;
}

PVX_POLY_FN int difficult_coeffs(const double *x) { // signed `biggest`, default branch
    double biggest = 0.0;
    for (int i = 0; i <= 4; i++)
        if (fabs(x[i]) > biggest) biggest = x[i];
    if (biggest == 0.0) return 0;
    for (int i = 0; i <= 4; i++)
        if (x[i] != 0.0 && fabs(biggest / x[i]) > 1.0e12) return 1;
    return 0;
}

PVX_POLY_FN int solve_quartic(const double *x, double *res) {
    double c1, c2, c3, c4, c0 = x[0];
    if (c0 != 1.0) {
        c1 = x[1] / c0; c2 = x[2] / c0; c3 = x[3] / c0; c4 = x[4] / c0;
    } else {
        c1 = x[1]; c2 = x[2]; c3 = x[3]; c4 = x[4];
    }
    double c12 = c1 * c1;
    double p = -0.375 * c12 + c2;
    double q = 0.125 * c12 * c1 - 0.5 * c1 * c2 + c3;
    double r = -0.01171875 * c12 * c12 + 0.0625 * c12 * c2 - 0.25 * c1 * c3 + c4;
    double cubic[4] = {1.0, -0.5 * p, -r, 0.5 * r * p - 0.125 * q * q};
    double roots[3];
    if (solve_cubic(cubic, roots) <= 0) return 0;
    double z = roots[0];
    double d1 = 2.0 * z - p, d2;
    if (d1 < 0.0) {
        if (d1 > -kSmall) d1 = 0.0;
        else return 0;
    }
    if (d1 < kSmall) {
        d2 = z * z - r;
        if (d2 < 0.0) return 0;
        d2 = sqrt(d2);
    } else {
        d1 = sqrt(d1);
        d2 = 0.5 * q / d1;
    }
    double q1 = d1 * d1, q2 = -0.25 * c1;
    double v[4];
    int i = 0;
    p = q1 - 4.0 * (z - d2);
    if (p == 0) {
        put_root(v, i, -0.5 * d1 - q2);
    } else if (p > 0) {
        p = sqrt(p);
        put_root(v, i, -0.5 * (d1 + p) + q2);
        put_root(v, i, -0.5 * (d1 - p) + q2);
    }
    p = q1 - 4.0 * (z + d2);
    if (p == 0) {
        put_root(v, i, 0.5 * d1 - q2);
    } else if (p > 0) {
        p = sqrt(p);
        put_root(v, i, 0.5 * (d1 + p) + q2);
        put_root(v, i, 0.5 * (d1 - p) + q2);
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (j < i) res[j] = v[j];
    return i;
}

// Solve_Polynomial for order 4 (polynomialsolver.cpp:1585-1732), c descending.
PVX_POLY_FN int solve4(const double *c0, double *r, bool sturm, double eps) {
    int i = 0, n = 4;
    while (i < n && fabs(c0[i]) < kSmall) i++;
    n -= i;
    const double *c = &c0[i];
    switch (n) {
    case 0:
        return 0;
    case 1:
        if (c[0] != 0.0) { r[0] = -c[1] / c[0]; return 1; }
        return 0;
    case 2:
        return solve_quadratic(c, r);
    case 3:
        if (eps > 0.0 && c[2] != 0.0 && fabs(c[3] / c[2]) < eps) return solve_quadratic(c, r);
        return sturm ? polysolve_n<3>(c, r) : solve_cubic(c, r);
    default:
        if (eps > 0.0 && c[3] != 0.0 && fabs(c[4] / c[3]) < eps)
            return sturm ? polysolve_n<3>(c, r) : solve_cubic(c, r);
        if (difficult_coeffs(c)) sturm = true;
        return sturm ? polysolve_n<4>(c, r) : solve_quartic(c, r);
    }
}

// Solve_Polynomial with epsilon 0 for orders up to 6 (the lathe's and sor's
// calls, lathe.cpp:255-285 and sor.cpp:395), c descending.
PVX_POLY_FN int solve6(int n, const double *c0, double *r, bool sturm) {
    int i = 0;
    while (i < n && fabs(c0[i]) < kSmall) i++;
    n -= i;
    const double *c = &c0[i];
    switch (n) {
    case 0:
        return 0;
    case 1:
        if (c[0] != 0.0) { r[0] = -c[1] / c[0]; return 1; }
        return 0;
    case 2:
        return solve_quadratic(c, r);
    case 3:
        return sturm ? polysolve_n<3>(c, r) : solve_cubic(c, r);
    case 4:
        if (difficult_coeffs(c)) sturm = true;
        return sturm ? polysolve_n<4>(c, r) : solve_quartic(c, r);
    default:
        return polysolve<6>(n, c, r);
    }
}
} // namespace poly

} // namespace pvx

#endif
