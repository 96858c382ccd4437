// Constants of the TNF pair model (the logistic models of cal_tnf_dist,
// cuda/Cuda2.cu:170-241 and 721-779) in the two forms the device uses.
//
// 1. The monomial coefficient tables, for the FP64 tie-breaker, which repeats
//    the reference's device arithmetic (cal_tnf_pre_dist_d).
// 2. A tensor Chebyshev re-expansion of each of the four polynomials
//    b1, c1, b2, c2 (x = min log size, y = max log size) on the square
//    [log10 1500, log10 500000]^2, for the FP32 evaluator.  In the monomial
//    basis the terms reach 1e8 while the values are 1..66, so FP32 evaluation
//    loses everything; in the Chebyshev basis sum |C| is O(100) and FP32 keeps
//    ~1e-5 absolute accuracy.  The expansion is computed once from the
//    monomial tables by exact-degree interpolation at Gauss-Chebyshev nodes in
//    x87 extended precision (degree <= 7 in x and <= 6 in y, so 8 x 7 nodes
//    reproduce each polynomial exactly up to rounding).
#include <cmath>
#include <cstring>
#include <vector>

#include "host_common.h"
#include "model_tables.h"

namespace mdet {

// Monomial exponents (px, py) of each coefficient, in the order of the
// reference's tables (cuda/Cuda2.cu:221-236 via the lw[] map of lines 201-219).
static const int EXP_B1[18][2] = {{0, 0}, {1, 0}, {0, 1}, {2, 0}, {0, 2}, {3, 0}, {0, 3}, {4, 0}, {0, 4},
                                  {5, 0}, {0, 5}, {6, 0}, {7, 0}, {1, 1}, {2, 2}, {3, 3}, {4, 4}, {5, 5}};
static const int EXP_B2[17][2] = {{0, 0}, {1, 0}, {0, 1}, {2, 0}, {0, 2}, {3, 0}, {0, 3}, {4, 0}, {0, 4},
                                  {5, 0}, {0, 5}, {6, 0}, {0, 6}, {2, 2}, {3, 3}, {4, 4}, {5, 5}};
static const int EXP_C2[19][2] = {{0, 0}, {1, 0}, {0, 1}, {2, 0}, {0, 2}, {3, 0}, {0, 3}, {4, 0}, {0, 4}, {5, 0},
                                  {0, 5}, {6, 0}, {0, 6}, {7, 0}, {1, 1}, {2, 2}, {3, 3}, {4, 4}, {5, 5}};

static long double eval_monomial(const double* coef, const int (*ex)[2], int nterm, long double x, long double y) {
    long double s = 0;
    for (int t = 0; t < nterm; ++t) {
        long double m = coef[t];
        for (int k = 0; k < ex[t][0]; ++k) m *= x;
        for (int k = 0; k < ex[t][1]; ++k) m *= y;
        s += m;
    }
    return s;
}

// Chebyshev coefficients (extended precision) of one monomial polynomial on
// the model square; exact up to rounding (degree <= 7 in x, <= 6 in y).
static void cheb_fit_ld(const double* coef, const int (*ex)[2], int nterm, long double out[MODEL_CX][MODEL_CY]) {
    const int NX = MODEL_CX, NY = MODEL_CY;
    const long double pi = 3.141592653589793238462643383279502884L;
    const long double lo = MODEL_XLO, hi = MODEL_XHI;
    const long double mid = 0.5L * (lo + hi), half = 0.5L * (hi - lo);
    long double f[NX][NY], tx[NX], ty[NY];
    for (int a = 0; a < NX; ++a) tx[a] = cosl(pi * (a + 0.5L) / NX);
    for (int b = 0; b < NY; ++b) ty[b] = cosl(pi * (b + 0.5L) / NY);
    for (int a = 0; a < NX; ++a)
        for (int b = 0; b < NY; ++b) f[a][b] = eval_monomial(coef, ex, nterm, mid + half * tx[a], mid + half * ty[b]);
    for (int p = 0; p < NX; ++p)
        for (int q = 0; q < NY; ++q) {
            long double acc = 0;
            for (int a = 0; a < NX; ++a)
                for (int b = 0; b < NY; ++b)
                    acc += f[a][b] * cosl(p * pi * (a + 0.5L) / NX) * cosl(q * pi * (b + 0.5L) / NY);
            acc *= (2.0L / NX) * (2.0L / NY);
            if (p == 0) acc *= 0.5L;
            if (q == 0) acc *= 0.5L;
            out[p][q] = acc;
        }
}

static void cheb_fit(const double* coef, const int (*ex)[2], int nterm, float out[MODEL_CX][MODEL_CY],
                     double* abs_sum) {
    long double C[MODEL_CX][MODEL_CY];
    cheb_fit_ld(coef, ex, nterm, C);
    double s = 0;
    for (int p = 0; p < MODEL_CX; ++p)
        for (int q = 0; q < MODEL_CY; ++q) {
            out[p][q] = (float)C[p][q];
            s += (double)fabsl(C[p][q]);
        }
    if (abs_sum) *abs_sum = s;
}

void model_cheb_tables(ModelCheb* m) {
    cheb_fit(kB1, EXP_B1, 18, m->c[0], &m->abs_sum[0]);
    cheb_fit(kC1, EXP_B1, 18, m->c[1], &m->abs_sum[1]);
    cheb_fit(kB2, EXP_B2, 17, m->c[2], &m->abs_sum[2]);
    cheb_fit(kC2, EXP_C2, 19, m->c[3], &m->abs_sum[3]);
}

// preProb of the full model (both logistic models, floor ln 9) at distance d,
// x = min and y = max log size, in extended precision.
static long double model_pre_ld(long double d, long double x, long double y) {
    long double b = eval_monomial(kB1, EXP_B1, 18, x, y), c = eval_monomial(kC1, EXP_B1, 18, x, y);
    long double pre = -(b + c * d);
    if (pre <= (long double)MODEL_FLOOR_PREPROB) {
        b = eval_monomial(kB2, EXP_B2, 17, x, y);
        c = eval_monomial(kC2, EXP_C2, 19, x, y);
        pre = -(b + c * d);
        if (pre > (long double)MODEL_FLOOR_PREPROB) pre = MODEL_FLOOR_PREPROB;
    }
    return pre;
}

// ---- proven upper bound of dthr over {xlo <= x <= y <= xhi} ----
//
// dthr of one model is g = N / c with N = -T' - b (T' = T, or ln 9 for the
// model-1 part below the floor), b and c the model's polynomials.  For a
// candidate t, "g <= t on the triangle" is "the polynomial N - t c is <= 0 and
// c > 0 there", which Bernstein coefficients decide: with y = xlo + h v and
// x = xlo + h s v (h = xhi - xlo) the triangle is the unit square of (s, v),
// b and c have degrees 7 and 10 there, and a polynomial on a cell lies between
// its smallest and largest Bernstein coefficient, whose corner entries are its
// values at the cell's corners.  Branch and bound: a cell all of whose
// coefficients have N - (best + tol/2) c <= 0 is dropped, `best` being the
// largest corner value of g seen; others are halved (de Casteljau, in turn
// along s and v).  The bound's gap shrinks with the square of the cell size,
// so a few hundred cells reach tol: 0.1-0.3 ms a radius measured on one host
// core, against 4-240 ms for second-order Taylor bounds per cell with global
// derivative bounds (Markov's inequality), most of an edge-list call on new
// contig lengths at 50,000 contigs (21 of 31 ms).  Rounding: the conversion
// runs in extended precision, the halvings are averages of doubles (error
// below 1e-11 for coefficients up to 1e3); the other tol/2 covers it.
namespace {

constexpr int BN_S = 8, BN_V = 11;  // Bernstein coefficients per variable (degrees 7 and 10)

struct Bern {
    double c[BN_V][BN_S];
};

// Bernstein form of a monomial polynomial on the triangle of [lo, lo + h].
Bern bern_of(const double* coef, const int (*ex)[2], int nterm, long double lo, long double h) {
    auto binom = [](int n, int k) {
        long double r = 1;
        for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
        return r;
    };
    // x = lo + h s v, y = lo + h v: coefficient of s^i v^m from x^a y^b is
    // C(a, i) C(b, m - i) lo^(a + b - m) h^m
    long double a[BN_V][BN_S] = {};
    for (int t = 0; t < nterm; ++t)
        for (int i = 0; i <= ex[t][0]; ++i)
            for (int j = 0; j <= ex[t][1]; ++j) {
                long double m = coef[t] * binom(ex[t][0], i) * binom(ex[t][1], j);
                for (int k = i + j; k < ex[t][0] + ex[t][1]; ++k) m *= lo;
                for (int k = 0; k < i + j; ++k) m *= h;
                a[i + j][i] += m;
            }
    Bern B;
    for (int m = 0; m < BN_V; ++m)
        for (int i = 0; i < BN_S; ++i) {
            long double v = 0;
            for (int q = 0; q <= m; ++q)
                for (int p = 0; p <= i; ++p)
                    v += binom(m, q) / binom(BN_V - 1, q) * (binom(i, p) / binom(BN_S - 1, p)) * a[q][p];
            B.c[m][i] = (double)v;
        }
    return B;
}

// The two halves of B along s or v.
void bern_halve(const Bern& B, bool along_v, Bern* lo, Bern* hi) {
    *hi = B;
    if (along_v) {
        for (int k = 0; k < BN_V; ++k) {
            for (int i = 0; i < BN_S; ++i) lo->c[k][i] = hi->c[0][i];
            for (int m = 0; m + 1 < BN_V - k; ++m)
                for (int i = 0; i < BN_S; ++i) hi->c[m][i] = 0.5 * (hi->c[m][i] + hi->c[m + 1][i]);
        }
    } else {
        for (int m = 0; m < BN_V; ++m)
            for (int k = 0; k < BN_S; ++k) {
                lo->c[m][k] = hi->c[m][0];
                for (int i = 0; i + 1 < BN_S - k; ++i) hi->c[m][i] = 0.5 * (hi->c[m][i] + hi->c[m][i + 1]);
            }
    }
}

struct Cell {
    Bern n, c;
    bool along_v;  // direction of the next halving
};

// An upper bound of max N / c over the triangle, at most tol above it; 1e30 if
// none is found (c not positive).
long double ratio_max(const Bern& N, const Bern& C, long double tol) {
    std::vector<Cell> work{Cell{N, C, true}};
    double best = -1e30;
    auto corners = [&](const Cell& q) {
        for (int m = 0; m < BN_V; m += BN_V - 1)
            for (int i = 0; i < BN_S; i += BN_S - 1) {
                if (!(q.c.c[m][i] > 0)) return false;
                best = std::fmax(best, q.n.c[m][i] / q.c.c[m][i]);
            }
        return true;
    };
    if (!corners(work[0])) return 1e30L;
    for (int cells = 0; !work.empty(); ++cells) {
        if (cells > 200000) return 1e30L;  // no convergence: the caller falls back
        const Cell q = work.back();
        work.pop_back();
        const double t = best + 0.5 * (double)tol;
        bool below = true;
        for (int m = 0; m < BN_V && below; ++m)
            for (int i = 0; i < BN_S; ++i) below &= q.n.c[m][i] - t * q.c.c[m][i] <= 0 && q.c.c[m][i] > 0;
        if (below) continue;
        Cell a, b;
        a.along_v = b.along_v = !q.along_v;
        bern_halve(q.n, q.along_v, &a.n, &b.n);
        bern_halve(q.c, q.along_v, &a.c, &b.c);
        if (!corners(a) || !corners(b)) return 1e30L;
        work.push_back(a);
        work.push_back(b);
    }
    return best + tol;
}

long double ratio_bound(const double* cb, const int (*eb)[2], int nb, const double* cc, const int (*ec)[2], int nc,
                        long double Tp, long double lo, long double hi, long double tol) {
    if (hi == lo) return (-Tp - eval_monomial(cb, eb, nb, lo, lo)) / eval_monomial(cc, ec, nc, lo, lo) + tol;
    Bern N = bern_of(cb, eb, nb, lo, hi - lo);
    for (auto& row : N.c)
        for (double& v : row) v = (double)(-Tp - (long double)v);
    return ratio_max(N, bern_of(cc, ec, nc, lo, hi - lo), tol);
}

}  // namespace

// Upper bound (proven, see above; within 1e-7 of the true maximum) over log
// sizes xlo <= x <= y <= xhi of the largest distance at which a pair can be an
// edge: model 1 passes up to d1 = (-T1 - b1)/c1, and, if model2, model 2 up
// to d2 = (-T2 - b2)/c2 (pairs whose model 1 is at or below ln 9).
double model_dthr_max(double xlo, double xhi, double T1, bool model2, double T2) {
    const long double lo = xlo, hi = xhi > xlo ? xhi : xlo;
    const long double tol = 1e-7L;
    long double m = ratio_bound(kB1, EXP_B1, 18, kC1, EXP_B1, 18, T1, lo, hi, tol);
    if (model2) m = fmaxl(m, ratio_bound(kB2, EXP_B2, 17, kC2, EXP_C2, 19, T2, lo, hi, tol));
    if (m >= 1e29L) m = 2.0L;  // no bound found: every pair of unit rows (d <= sqrt 2) passes
    return (double)m;
}

// Threshold preProb > T (gen_tnf_graph): model 1 above max(T, ln 9); model 2
// only if T < ln 9 (its value is clamped to ln 9, which never exceeds T >= ln 9).
double model_dthr_max(double xlo, double xhi, double T) {
    const double fl = MODEL_FLOOR_PREPROB;
    return model_dthr_max(xlo, xhi, T >= fl ? T : fl, T < fl, T);
}

double model_pre_reference(double d, double x, double y) { return (double)model_pre_ld(d, x, y); }

}  // namespace mdet

extern "C" {

int mdet_model_radius(double xlo, double xhi, double cutoff, double* radius) {
    if (!radius) MDET_FAIL(MDET_E_INVALID, "mdet_model_radius: null output");
    if (!(cutoff > 0 && cutoff < 1)) MDET_FAIL(MDET_E_INVALID, "mdet_model_radius: cutoff %g not in (0, 1)", cutoff);
    const double lo = std::log10(1500.0), hi = std::log10(500000.0);
    if (!(xlo >= lo - 1e-12 && xhi <= hi + 1e-12 && xlo <= xhi))
        MDET_FAIL(MDET_E_RANGE, "mdet_model_radius: log sizes [%g, %g] outside [log10 1500, log10 500000]", xlo, xhi);
    *radius = mdet::model_dthr_max(xlo, xhi, std::log((1.0 / (1.0 - cutoff)) - 1.0));
    return MDET_OK;
}

// Chebyshev coefficients of b1, c1, b2, c2 (4 x MODEL_CX x MODEL_CY floats,
// row p = degree in the min-size variable) for tests and the device upload.
int mdet_model_cheb(float* out, double* abs_sum4, double* domain2) {
    if (!out) MDET_FAIL(MDET_E_INVALID, "mdet_model_cheb: null output");
    mdet::ModelCheb m;
    mdet::model_cheb_tables(&m);
    memcpy(out, m.c, sizeof m.c);
    if (abs_sum4)
        for (int i = 0; i < 4; ++i) abs_sum4[i] = m.abs_sum[i];
    if (domain2) {
        domain2[0] = MODEL_XLO;
        domain2[1] = MODEL_XHI;
    }
    return MDET_OK;
}

// The monomial coefficient table `which` (0 b1, 1 c1, 2 b2, 3 c2) the library
// evaluates, with each term's exponents (x = min, y = max log size).
int mdet_model_coefs(int which, double* coef, int32_t* exps_xy, uint32_t cap, uint32_t* count) {
    if (which < 0 || which > 3 || !count) MDET_FAIL(MDET_E_INVALID, "mdet_model_coefs: bad table %d", which);
    static const double* tabs[4] = {mdet::kB1, mdet::kC1, mdet::kB2, mdet::kC2};
    static const int nterm[4] = {18, 18, 17, 19};
    const int(*ex)[2] = which < 2 ? mdet::EXP_B1 : which == 2 ? mdet::EXP_B2 : mdet::EXP_C2;
    *count = (uint32_t)nterm[which];
    if (cap < (uint32_t)nterm[which])
        MDET_FAIL(MDET_E_CAPACITY, "mdet_model_coefs: table %d has %d terms", which, nterm[which]);
    for (int t = 0; t < nterm[which]; ++t) {
        if (coef) coef[t] = tabs[which][t];
        if (exps_xy) {
            exps_xy[2 * t] = ex[t][0];
            exps_xy[2 * t + 1] = ex[t][1];
        }
    }
    return MDET_OK;
}

}  // extern "C"
