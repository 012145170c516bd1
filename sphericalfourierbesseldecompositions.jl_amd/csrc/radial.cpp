// A common radial basis for every spline of a plan: clamped B-splines of degree 9 on one set
// of breaks, and each map's g_nl as a combination of them (host setup of the mixed path).
//
// A catalogue then needs spreading onto the basis' ~160 functions only, instead of one map
// per (n, l).  The breaks follow what the splines resolve: 20 knot spacings of the finest
// one in the middle (the reference takes ~24 knots per period of g_nl, so a degree-9 basis at
// that spacing represents the smooth part to ~1e-9), graded down by 1.3 to half a spacing
// towards both ends, where every natural cubic spline has a boundary layer of a few of its
// own spacings.  What remains is the splines' own interpolation error (third derivatives jump
// at every knot): 5e-9 of a spline's largest value, 1.3e-8 at most for the reference's knots.
// Tables that are not represented to RADIAL_TOL keep the per-map path.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <exception>
#include <new>
#include <thread>

#include "sfb_internal.h"

namespace sfb {

namespace {

constexpr int P = RADIAL_DEGREE;
constexpr double MIDDLE = 20.0, FINEST = 0.5, GRADE = 1.3;  // in knot spacings; growth per interval
constexpr int SAMPLES = 32;  // fit points per interval (a middle interval holds ~20 knots)
constexpr int CHECKS = 11;   // check points per interval, between the fit points

// The P + 1 B-splines that are non-zero on [t[P+iv], t[P+iv+1]] at x (Cox-de Boor).
void bspline(const std::vector<double>& t, int iv, double x, double* out)
{
    double left[P + 1], right[P + 1];
    const int i = P + iv;
    out[0] = 1.0;
    for (int k = 1; k <= P; ++k) {
        left[k] = x - t[(size_t)(i + 1 - k)];
        right[k] = t[(size_t)(i + k)] - x;
        double saved = 0.0;
        for (int j = 0; j < k; ++j) {
            const double tmp = out[j] / (right[j + 1] + left[k - j]);
            out[j] = saved + right[j + 1] * tmp;
            saved = left[k - j] * tmp;
        }
        out[k] = saved;
    }
}

}  // namespace

static bool fit(int64_t nmaps, const int64_t* off, const double* kx, const double* ky, const double* kypp,
                RadialBasis* R, int threads)
{
    if (nmaps < 1) return false;
    for (int64_t q = 0; q < nmaps; ++q)  // (this runs beside the plan's own checks of the tables)
        if (off[q + 1] - off[q] < 4) return false;
    const double lo = kx[off[0]], hi = kx[off[1] - 1];
    double H = hi - lo;
    for (int64_t q = 0; q < nmaps; ++q) {
        const int64_t nk = off[q + 1] - off[q];
        if (kx[off[q]] != lo || kx[off[q + 1] - 1] != hi) return false;
        H = std::min(H, (hi - lo) / (double)(nk - 1));
    }
    const double len = hi - lo;
    if (!(len > 0.0) || !std::isfinite(len) || !(H > 0.0)) return false;
    // breaks of the lower half, then mirrored
    std::vector<double> half(1, 0.0);
    while (half.back() < 0.5 * len) {
        if ((int64_t)half.size() > RADIAL_MAX) return false;
        half.push_back(half.back() + std::min(MIDDLE * H, std::max(FINEST * H, (GRADE - 1.0) * half.back())));
    }
    const double sc = 0.5 * len / half.back();
    std::vector<double> brk;
    for (double v : half) brk.push_back(lo + sc * v);
    for (size_t i = half.size() - 1; i-- > 0;) brk.push_back(i == 0 ? hi : hi - sc * half[i]);
    const int niv = (int)brk.size() - 1, nc = niv + P;
    if (nc > RADIAL_MAX) return false;
    for (int i = 0; i < niv; ++i)
        if (!(brk[(size_t)i + 1] > brk[(size_t)i])) return false;
    std::vector<double> t((size_t)P, lo);
    t.insert(t.end(), brk.begin(), brk.end());
    t.insert(t.end(), (size_t)P, hi);
    // fit and check points, in increasing order, with their basis values
    struct Pt { double x; int iv; double w; double b[P + 1]; };
    std::vector<Pt> pts;
    auto add = [&](double x, int iv, double w) {
        Pt p;
        p.x = x;
        p.iv = iv;
        p.w = w;
        bspline(t, iv, x, p.b);
        pts.push_back(p);
    };
    for (int iv = 0; iv < niv; ++iv) {
        const double a = brk[(size_t)iv], d = brk[(size_t)iv + 1] - a;
        if (iv == 0) add(lo, 0, 16.0);
        std::vector<std::pair<double, double>> u;
        for (int s = 0; s < SAMPLES; ++s) u.push_back({(s + 0.5) / SAMPLES, 1.0});
        for (int s = 0; s < CHECKS; ++s) u.push_back({(s + 1.0) / (CHECKS + 1.0), 0.0});
        std::sort(u.begin(), u.end());
        for (auto& v : u) add(a + d * v.first, iv, v.second);
        if (iv == niv - 1) add(hi, niv - 1, 16.0);
    }
    // normal equations B^T W B (banded, lower, column j holds rows j .. j + P): Cholesky
    const int W = P + 1;
    std::vector<double> G((size_t)nc * W, 0.0);
    for (const Pt& p : pts)
        for (int a = 0; a <= P && p.w > 0.0; ++a)
            for (int b = a; b <= P; ++b) G[(size_t)(p.iv + a) * W + (b - a)] += p.w * p.b[a] * p.b[b];
    for (int j = 0; j < nc; ++j) {
        double* gj = G.data() + (size_t)j * W;
        for (int k = std::max(0, j - P); k < j; ++k) {
            const double* gk = G.data() + (size_t)k * W;
            const double f = gk[j - k];
            for (int i = 0; i + j - k < W; ++i) gj[i] -= f * gk[i + j - k];
        }
        if (!(gj[0] > 0.0)) return false;
        const double d = 1.0 / std::sqrt(gj[0]);
        for (int i = 0; i < W; ++i) gj[i] *= d;
    }
    R->nc = nc;
    R->niv = niv;
    R->t = t;
    R->gamma.assign((size_t)nmaps * nc, 0.0);
    std::atomic<int64_t> next{0};
    std::atomic<bool> good{true};
    std::vector<double> worst((size_t)nmaps, 0.0);
    auto work = [&]() {
        std::vector<double> val;
        try {
            val.resize(pts.size());
        } catch (const std::bad_alloc&) {
            good = false;
            return;
        }
        for (int64_t q; (q = next.fetch_add(1)) < nmaps;) {
            const int64_t o = off[q], nk = off[q + 1] - off[q];
            const double *x = kx + o, *y = ky + o, *m = kypp + o;
            double big = 0.0;
            int64_t i = 0;
            double* c = R->gamma.data() + (size_t)q * nc;
            for (size_t e = 0; e < pts.size(); ++e) {
                const Pt& p = pts[e];
                while (i + 2 < nk && x[i + 1] <= p.x) ++i;
                const double h = x[i + 1] - x[i], u = (p.x - x[i]) / h, h2 = h * h;
                const double b = 0.5 * h2 * m[i], a = h2 * (m[i + 1] - m[i]) / 6.0;
                const double v = y[i] + u * (y[i + 1] - a - b - y[i] + u * (b + u * a));
                val[e] = v;
                big = std::max(big, std::fabs(v));
                if (p.w > 0.0)
                    for (int s = 0; s <= P; ++s) c[p.iv + s] += p.w * p.b[s] * v;
            }
            for (int j = 0; j < nc; ++j) {  // L z = rhs
                double v = c[j];
                for (int k = std::max(0, j - P); k < j; ++k) v -= G[(size_t)k * W + (j - k)] * c[k];
                c[j] = v / G[(size_t)j * W];
            }
            for (int j = nc - 1; j >= 0; --j) {  // L^T c = z
                double v = c[j];
                for (int k = j + 1; k <= std::min(nc - 1, j + P); ++k) v -= G[(size_t)j * W + (k - j)] * c[k];
                c[j] = v / G[(size_t)j * W];
            }
            double err = 0.0;
            for (size_t e = 0; e < pts.size(); ++e) {
                const Pt& p = pts[e];
                double f = 0.0;
                for (int s = 0; s <= P; ++s) f += p.b[s] * c[p.iv + s];
                err = std::max(err, std::fabs(f - val[e]));
            }
            worst[(size_t)q] = big > 0.0 ? err / big : 0.0;
            if (!(err <= RADIAL_TOL * big)) {  // also catches NaN
                good = false;
                next = nmaps;
            }
        }
    };
    const int nt = (int)std::min<int64_t>(std::max(1, threads), 1 + nmaps / 16);
    std::vector<std::thread> th;
    th.reserve((size_t)nt);  // (a failure here leaves no thread behind)
    try {
        for (int i = 1; i < nt; ++i) th.emplace_back(work);
    } catch (const std::exception&) {  // no thread or no memory for one: the others do the rest
    }
    work();
    for (std::thread& x : th) x.join();
    R->err = *std::max_element(worst.begin(), worst.end());
    return good;
}

bool radial_basis(int64_t nmaps, const int64_t* off, const double* kx, const double* ky, const double* kypp,
                  RadialBasis* R, int threads)
{
    try {
        return fit(nmaps, off, kx, ky, kypp, R, threads);
    } catch (const std::bad_alloc&) {  // without the basis the plan keeps the per-map path
        return false;
    }
}

}  // namespace sfb
