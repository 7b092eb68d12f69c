// Per-lane body of the primary-Compton scatter kernels.
//
// Reference: crystalScatterSysMatCuda and collimatorScatterSysMatCuda
// (ScatterGen_RayTracing_CircularHole/scatter.cu:1077-1437, :1544-1936;
// standalone variant ScatterGen_Collimator/scatter.cu:1056-1435).  One term is
// (voxel v, scatter point s, detection sub-cell of bar d):
//
//   w_s(v) * Phi/(2 pi) * K(theta_min, theta_max) * P_E * exp(-att2) * abs'
//
// The second-leg attenuation runs from s to the sub-cell, so its chords do
// not depend on v; only the energy scaling does, through E'(theta(v)):
//   att2 = (E0/E')^3 * S_pe + (E0/E') * S_c,
//   S_pe = sum_k l_k mu_pe_k + (l1 - l2) mu_pe_d,  S_c likewise with mu_c,
// the same sum the reference forms term by term (scatter.cu:1343-1417).
// S_pe, S_c, the absorption chord and |s - q| are computed once per
// (d, s, sub-cell) by the FP64 pair-terms kernel and read here.
#pragma once

#include <cmath>

#include "smg_pe_body.hpp"

namespace smg {

struct PairTerm {
    double s_pe, s_c, la, len;  // len = |scatter point - sub-cell centre|
    double s_wpe, s_wc;         // collimator material on the second leg (grid scatterers)
};

// The record the pair-terms kernel writes per (row, scatter point, sub-cell):
// the pair terms, and 1 / |corner - scatter point| for the sub-cell's 8 corners
// (corner c has lo[k] or hi[k] on axis k as bit k of c is clear or set), which
// the polar range of every voxel's term shares.
struct PairRec {
    PairTerm t;
    double ic[8];
};

// 1 / |corner c - qss| of the box [lo, hi].
SMG_FN double inv_corner(const double lo[3], const double hi[3], const double qss[3], int c) {
    double w2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double w = ((c >> k) & 1 ? hi[k] : lo[k]) - qss[k];
        w2 += w * w;
    }
    return 1.0 / sqrt(w2);
}

// ---- collimator material for grid scatterers ----------------------------------------
// (An extension with no reference counterpart.)  Plain intersection lengths of
// a segment with a box and with a finite cylinder along y, without the
// reference chord functions' thresholds, in FP64.

SMG_FN double seg_box_geo(const double a[3], const double b[3], const double lo[3],
                          const double hi[3]) {
    double t0 = 0.0, t1 = 1.0;
    for (int k = 0; k < 3; ++k) {
        const double D = b[k] - a[k];
        if (D == 0.0) {
            if (a[k] < lo[k] || a[k] > hi[k]) return 0.0;
            continue;
        }
        double u = (lo[k] - a[k]) / D, w = (hi[k] - a[k]) / D;
        if (u > w) {
            const double x = u;
            u = w;
            w = x;
        }
        t0 = tmax2(t0, u);
        t1 = tmin2(t1, w);
    }
    if (!(t1 > t0)) return 0.0;
    const double dx = b[0] - a[0], dy = b[1] - a[1], dz = b[2] - a[2];
    return (t1 - t0) * sqrt(dx * dx + dy * dy + dz * dz);
}

// Fraction of the segment a -> b (its parameter range in [0, 1]) inside the
// cylinder of radius r about the line x = xc, z = zc, for y1 <= y <= y2.
SMG_FN double seg_cyl_frac(const double a[3], const double b[3], double xc, double y1, double y2,
                           double zc, double r) {
    const double D[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
    double t0 = 0.0, t1 = 1.0;
    if (D[1] == 0.0) {
        if (a[1] < y1 || a[1] > y2) return 0.0;
    } else {
        double u = (y1 - a[1]) / D[1], w = (y2 - a[1]) / D[1];
        if (u > w) {
            const double x = u;
            u = w;
            w = x;
        }
        t0 = tmax2(t0, u);
        t1 = tmin2(t1, w);
    }
    const double x0 = a[0] - xc, z0 = a[2] - zc;
    const double A = D[0] * D[0] + D[2] * D[2], B = x0 * D[0] + z0 * D[2],
                 Cq = x0 * x0 + z0 * z0 - r * r;
    if (A == 0.0) {
        if (Cq > 0.0) return 0.0;
    } else {
        const double disc = B * B - A * Cq;
        if (disc <= 0.0) return 0.0;
        const double sq = sqrt(disc);
        t0 = tmax2(t0, (-B - sq) / A);
        t1 = tmin2(t1, (-B + sq) / A);
    }
    return t1 > t0 ? t1 - t0 : 0.0;
}

SMG_FN double seg_cyl_geo(const double a[3], const double b[3], double xc, double y1, double y2,
                          double zc, double r) {
    const double f = seg_cyl_frac(a, b, xc, y1, y2, zc, r);
    if (!(f > 0.0)) return 0.0;
    const double D[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
    return f * sqrt(D[0] * D[0] + D[1] * D[1] + D[2] * D[2]);
}

// Elliptical hole o (semi-axes erx, erz along x', z', the (x, z) offsets from
// the axis turned by theta): in the coordinates x'/erx, z'/erz its section is
// the unit circle.  That map is linear, so a segment's parameter range inside
// is the mapped segment's range inside the unit cylinder.
SMG_FN double seg_ell_geo(const double a[3], const double b[3], const Hole<double>& o) {
    const double ax = a[0] - o.xc, az = a[2] - o.zc, bx = b[0] - o.xc, bz = b[2] - o.zc;
    const double am[3] = {(ax * o.ec + az * o.es) / o.erx, a[1], (-ax * o.es + az * o.ec) / o.erz};
    const double bm[3] = {(bx * o.ec + bz * o.es) / o.erx, b[1], (-bx * o.es + bz * o.ec) / o.erz};
    const double f = seg_cyl_frac(am, bm, 0.0, o.y1, o.y2, 0.0, 1.0);
    if (!(f > 0.0)) return 0.0;
    const double D[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
    return f * sqrt(D[0] * D[0] + D[1] * D[1] + D[2] * D[2]);
}

// Collimator material along a -> b at E0: each layer's plate chord less the
// chords of its holes (at least 0) with the layer's mu, plus the holes' own
// mu.  att_t: sum of mu_total l; s_pe, s_c: sums with the photoelectric and
// Compton coefficients.
SMG_FN void coll_material(const PeGeom& G, const double a[3], const double b[3], double& att_t,
                          double& s_pe, double& s_c) {
    att_t = s_pe = s_c = 0.0;
    for (int m = 0; m < G.g.n_layers; ++m) {
        const Layer<double>& L = G.layers_d[m];
        const double c = seg_box_geo(a, b, L.lo, L.hi);
        if (!(c > 0.0)) continue;  // a hole of the layer lies inside its plate box
        double holes = 0.0;
        const int first = G.g.ranges[m].first, last = first + G.g.ranges[m].count;
        for (int h = first; h < last; ++h) {
            const Hole<double>& o = G.holes_d[h];
            const double l = o.erx > 0.0 ? seg_ell_geo(a, b, o) : seg_cyl_geo(a, b, o.xc, o.y1, o.y2, o.zc, o.r);
            holes += l;
            att_t += o.mu * l;
            s_pe += o.mupe * l;
            s_c += o.muc * l;
        }
        const double wl = tmax2(c - holes, 0.0);
        att_t += L.mu * wl;
        s_pe += L.mupe * wl;
        s_c += L.muc * wl;
    }
}

// mu(E) tables (an extension with no reference counterpart): per process
// (0 crystal photoelectric, 1 crystal Compton, 2 collimator photoelectric,
// 3 collimator Compton) log mu on increasing log-energy nodes, linear in
// (log E, log mu) between nodes and continuing the end segments beyond them;
// lmu0 holds each table at E0.  n = 0: the reference's power laws.
constexpr int kMaxMuNodes = 256;
struct MuTables {
    int n;
    double le[kMaxMuNodes];
    double lmu[4][kMaxMuNodes];
    double lmu0[4];
};

SMG_FN double mu_table_log(const MuTables& t, int which, double le) {
    int lo = 0, hi = t.n - 1;
    while (hi - lo > 1) {  // the last node not above le, within [0, n - 2]
        const int mid = (lo + hi) >> 1;
        if (t.le[mid] <= le) lo = mid;
        else hi = mid;
    }
    const double f = (le - t.le[lo]) / (t.le[lo + 1] - t.le[lo]);
    return t.lmu[which][lo] + f * (t.lmu[which][lo + 1] - t.lmu[which][lo]);
}

// mu(E')/mu(E0) of the photoelectric (r3) and Compton (r1) processes of the
// crystal: the tables when given, else (E0/E')^3 and E0/E' (scatter.cu:1371-1375).
SMG_FN void mu_ratios(const MuTables* t, double e0, double ep, double& r3, double& r1) {
    if (!t || t->n == 0) {
        r1 = e0 / ep;
        r3 = e0 * e0 * e0 / ep / ep / ep;
        return;
    }
    const double le = log(ep);
    r3 = exp(mu_table_log(*t, 0, le) - t->lmu0[0]);
    r1 = exp(mu_table_log(*t, 1, le) - t->lmu0[1]);
}

// The tables in the form the FP32 term evaluates them.  E' lies in
// [E0 / (1 + 2 alpha), E0], so each process's ratio mu(E')/mu(E0) is a
// piecewise power law in L = ln(E0/E') on the few table segments that range
// meets: on segment j, ln(mu(E')/mu(E0)) = c[p][j] - s[p][j] L, with lb the
// segment breakpoints in L (ascending).  The FP32 term forms L from
// E0/E' = 1 + alpha (1 - cos theta) and needs no FP64 log or exp: its ratios
// are good to ~3e-7 relative (the FP64 term keeps the table search in FP64).
// n = 0: not available (too many segments in range); the FP32 term then
// takes the FP64 form.
constexpr int kMaxMuSegF = 24;
struct MuTablesF {
    int n;                       // segments
    float lb[kMaxMuSegF];        // lb[j], j < n - 1: upper end of segment j in L
    float c[4][kMaxMuSegF];
    float s[4][kMaxMuSegF];
};

// Segment of L (branch-free count of the breakpoints below it).
SMG_FN int mu_seg_f(const MuTablesF& t, float L) {
    int j = 0;
    for (int k = 0; k < t.n - 1; ++k) j += L > t.lb[k];
    return j;
}

SMG_FN float mu_ratio_f(const MuTablesF& t, int which, int j, float L) {
    const float x = t.c[which][j] - t.s[which][j] * L;
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_exp2f(x * 1.44269504088896341f);  // |x| is a few units: no denormals
#else
    return expf(x);
#endif
}

// ln(x) for x >= 1 not far above it (E0/E').
SMG_FN float log_f(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_logf(x) * 0.693147180559945309f;  // log2, normal argument
#else
    return logf(x);
#endif
}

// Host: the FP32 form of t for photopeak e0 (alpha = e0 / 511).
inline void make_mu_tables_f(const MuTables& t, double e0, MuTablesF& f) {
    f.n = 0;
    if (t.n < 2) return;
    const double alpha = e0 / 511.0, lmax = std::log(1.0 + 2.0 * alpha) * (1.0 + 1e-6), le0 = std::log(e0);
    double br[kMaxMuNodes];
    int nb = 0;
    for (int k = t.n - 1; k >= 0; --k) {  // nodes inside (E0 e^-lmax, E0), ascending in L
        const double L = le0 - t.le[k];
        if (L > 0.0 && L < lmax) br[nb++] = L;
    }
    if (nb + 1 > kMaxMuSegF) return;
    for (int j = 0; j <= nb; ++j) {
        const double a = j == 0 ? 0.0 : br[j - 1], b = j == nb ? lmax : br[j];
        const double le = le0 - 0.5 * (a + b);  // inside segment j
        int lo = 0, hi = t.n - 1;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (t.le[mid] <= le) lo = mid;
            else hi = mid;
        }
        if (j < nb) f.lb[j] = float(br[j]);
        for (int p = 0; p < 4; ++p) {
            const double slope = (t.lmu[p][lo + 1] - t.lmu[p][lo]) / (t.le[lo + 1] - t.le[lo]);
            f.c[p][j] = float(t.lmu[p][lo] + slope * (le0 - t.le[lo]) - t.lmu0[p]);
            f.s[p][j] = float(slope);
        }
    }
    f.n = nb + 1;
}

struct ScatterPhys {
    double e0, lo, hi;     // photopeak energy and energy window (keV)
    double norm;           // sum of KN sin over [0, pi] (scatter.cu:1169)
    double res;            // energy resolution of bar d at E0
    double rcell;          // bounding radius of a detection sub-cell
    double mupe, muc;      // bar d
    const MuTables* tab = nullptr;  // mu(E) tables, or power laws
    const MuTablesF* tabf = nullptr;  // their FP32 form (FP32 term), or none
    const double* knt = nullptr;    // KN prefix table (kn_sum_table), or the node loop: without
                                    // kTab only, which no kernel uses
    double c_rej = -2.0;            // cos(theta) below this is outside the window for
                                    // sure (window_reject_cos with the path's margin)
    // the kernels' tables (scatter_term with kTab set)
    const double* knp = nullptr;    // KN prefix polynomials (kn_poly_sum)
    double inv_norm = 0.0;          // 1 / norm
    const float* win = nullptr;     // window probability of the row (win_table_value), FP32
    double win_x0 = 0.0, win_scale = 0.0;  // its first 1 - cos(theta) and intervals per unit of it
    int win_n = 0;                  // its intervals
    double omc_lo = 3.0, omc_hi = -1.0;    // terms with 1 - cos(theta) >= omc_lo lie below the
                                    // window, those <= omc_hi above it
};

// Thresholds with their reference values.
constexpr double kFwhm = (double)2.35482f;  // scatter.cu:1026, :1263
constexpr double kKnStep = (double)0.01f;   // scatter.cu:1338 (0.01 passed as float)
constexpr double kTwoPi = 2.0 * 3.14159265358979323846;

// The lower 2-sigma window test of a term (scatter.cu:1263-1269) rejects it
// when e0 g (1 + res sqrt(g) 2/FWHM) <= lo, g = E'/E0 = 1 / (1 + alpha (1 -
// cos theta)).  The left side increases with g and g with cos theta, so the
// test is cos theta <= c_lo for one c_lo per (E0, window, bar resolution),
// found here by bisection in FP64.  Returns c_lo less `margin`, which covers
// the rounding of the cosine the caller compares (FP32: below 1e-6 for the
// unit vectors of a term, margin 1e-5; FP64: the reference's acos/cos round
// trip, margin 1e-9), so a term below it is rejected by the full test too;
// -2 when nothing is rejected.
SMG_FN double window_reject_cos(const ScatterPhys& ph, double margin) {
    const double alpha = ph.e0 / 511.0, r = ph.res * (2.0 / kFwhm);
    if (!(ph.lo > 0.0) || !(alpha > 0.0)) return -2.0;
    if (ph.e0 * (1.0 + r) <= ph.lo) return 2.0;  // every term is below the window
    double g0 = 0.0, g1 = 1.0;  // e0 g (1 + r sqrt g) <= lo at g0, > lo at g1
    for (int it = 0; it < 80; ++it) {
        const double gm = 0.5 * (g0 + g1);
        if (ph.e0 * gm * (1.0 + r * sqrt(gm)) <= ph.lo) g0 = gm;
        else g1 = gm;
    }
    const double c_lo = 1.0 - (1.0 / g0 - 1.0) / alpha;
    if (c_lo < -1.5) return -2.0;
    return c_lo - margin;
}

// window_reject_cos(ph, margin) from its value at margin 0: the special
// values -2 (nothing rejected) and 2 (everything rejected) carry no margin.
SMG_FN double window_cut_margin(double cut, double margin) {
    return (cut < -1.5 || cut > 1.5) ? cut : cut - margin;
}

// Klein-Nishina in the reference's factorised form (scatter.cu:962-977), from
// cos(theta).
template <class T>
SMG_FN T kn_of_cos(T c, T alpha) {
    T f1 = alpha * (T(1) - c);
    T f2 = T(1) + c * c;
    return f2 / (T(1) + f1) / (T(1) + f1) * (T(1) + f1 * f1 / f2 / (T(1) + f1));
}

// Inclusive rectangle rule of KN sin on lo + i*step, i = 0..n with
// n = (int)((hi - lo)/step) (scatter.cu:980-993).  FP32: flags a step count
// within rounding distance of an integer, and takes cos and sin of the nodes
// from an angle-addition recurrence in FP64 started at the FP32 cos and sin of
// lo (four FMAs a step instead of two transcendental calls; the rotation keeps
// the start's ~1e-7 error and drifts by about one FP64 ulp per step).  FP64:
// cos and sin of every node, as the reference.
template <class T>
SMG_FN T kn_sum(T lo, T hi, T alpha, bool& near) {
    const T step = T(kKnStep);
    T x = (hi - lo) / step;
    int n = (int)x;
    if constexpr (kGuarded<T>) {
        T fr = x - T(n);
        near |= (fr < T(2e-4) && n > 0) | (fr > T(1) - T(2e-4));
        // cos and sin of the step (double)0.01f = 0.009999999776482582
        const double cst = 0.99995000041890041468, snt = 0.0099998331106604225523;
        // start values in FP32 (the sum is FP32): an FP64 cos/sin here costs
        // more registers than the whole FP32 term
        float cf, sf;
        sincosf(float(lo), &sf, &cf);
        double c = cf, sv = sf;
        KahanSum<T> s;
        for (int i = 0; i <= n; ++i) {
            s.add(kn_of_cos(T(c), alpha) * T(sv) * step);
            const double c2 = c * cst - sv * snt;
            sv = sv * cst + c * snt;
            c = c2;
        }
        return s.value();
    } else {
        KahanSum<T> s;
        for (int i = 0; i <= n; ++i) {
            T th = lo + T(i) * step;
            T c = cos(th), sn = sin(th);
            s.add(kn_of_cos(c, alpha) * sn * step);
        }
        return s.value();
    }
}

// KN rectangle sums from a prefix table, which the host tests use: the kernels
// take the polynomials below.  The reference's sum has nodes
// lo + i step, i = 0..n; with lo = phi + k0 step (0 <= phi < step) it is
// P(phi, k0 + n) - P(phi, k0 - 1), P(phi, k) = sum_{i <= k} g(phi + i step),
// g(t) = KN(cos t) sin t step.  The table holds P in FP64 for kKnPhase + 1
// phases phi_j = j step / kKnPhase (rows) and k < kKnSteps nodes (columns);
// the sum is interpolated linearly in phi between rows j and j + 1 (error
// ~(step / kKnPhase)^2 / 8 times the sum's second derivative, ~1e-9 relative).
constexpr int kKnPhase = 256;
constexpr int kKnSteps = 320;  // nodes up to 3.19 rad; polar angles stay below pi

// Row j of the table for alpha = E0 / 511 (FP64, two-sum compensated).
SMG_FN void kn_prefix_row(double alpha, int j, double* row) {
    const double step = kKnStep;
    const double phi = step * (double)j / (double)kKnPhase;
    KahanSum<double> s;
    for (int k = 0; k < kKnSteps; ++k) {
        const double th = phi + (double)k * step;
        s.add(kn_of_cos<double>(cos(th), alpha) * sin(th) * step);
        row[k] = s.value();
    }
}

// The rectangle sum over [lo, hi] from the table; n as the FP32 node loop
// forms it (with the same near-integer flag).  A node range outside the
// table flags the term for FP64.
SMG_FN double kn_sum_table(const double* tab, float lo, float hi, bool& near) {
    const float stepf = float(kKnStep);
    const float x = (hi - lo) / stepf;
    const int n = (int)x;
    const float fr = x - float(n);
    near |= (fr < 2e-4f && n > 0) | (fr > 1.0f - 2e-4f);
    const double u = (double)lo * (1.0 / kKnStep);
    const int k0 = (int)floor(u);
    double ph = (u - (double)k0) * kKnPhase;
    int j = (int)ph;
    if (j >= kKnPhase) j = kKnPhase - 1;
    if (j < 0) j = 0;
    const double w = ph - (double)j;
    const int k1 = k0 + n;
    if (k0 < 0 || k1 >= kKnSteps) {
        near = true;
        return 0.0;
    }
    const double* r0 = tab + (size_t)j * kKnSteps;
    const double* r1 = r0 + kKnSteps;
    const double a0 = r0[k1] - (k0 > 0 ? r0[k0 - 1] : 0.0);
    const double a1 = r1[k1] - (k0 > 0 ? r1[k0 - 1] : 0.0);
    return a0 + w * (a1 - a0);
}

// KN rectangle sums from prefix polynomials.  P(phi, k) above is smooth in phi
// for every k: over phi = t step, 0 <= t < 1, it is held as a polynomial of degree
// kKnDeg through its values at the Chebyshev points of [0, 1], kKnStride doubles
// per k.  The truncation is below FP64 rounding (the step is 0.01 rad), so a sum
// is good to ~1e-15 absolute; 20 KB stay in a compute unit's first-level cache,
// where the 658 KB table of phases (kn_prefix_row) was read from the second level.
constexpr int kKnDeg = 6;
constexpr int kKnStride = 8;
constexpr int kKnPolySize = kKnSteps * kKnStride;

// Chebyshev point m of kKnDeg + 1 on [0, 1].
SMG_FN double kn_phase(int m) {
    return 0.5 * (1.0 - cos(3.14159265358979323846 * (2 * m + 1) / (2.0 * (kKnDeg + 1))));
}
// Node k of phase t (in steps): KN sin times the step.
SMG_FN double kn_node(double alpha, double t, int k) {
    const double th = (t + (double)k) * kKnStep;
    return kn_of_cos<double>(cos(th), alpha) * sin(th) * kKnStep;
}
// Power coefficients of the polynomial with the values v at the points kn_phase
// (Newton's divided differences, expanded).
SMG_FN void kn_poly_coeffs(const double v[kKnDeg + 1], double c[kKnDeg + 1]) {
    double d[kKnDeg + 1], x[kKnDeg + 1];
    for (int i = 0; i <= kKnDeg; ++i) {
        d[i] = v[i];
        x[i] = kn_phase(i);
        c[i] = 0.0;
    }
    for (int j = 1; j <= kKnDeg; ++j)
        for (int i = kKnDeg; i >= j; --i) d[i] = (d[i] - d[i - 1]) / (x[i] - x[i - j]);
    for (int i = kKnDeg; i >= 0; --i) {  // c <- c (t - x_i) + d_i
        for (int j = kKnDeg; j >= 1; --j) c[j] = c[j - 1] - x[i] * c[j];
        c[0] = d[i] - x[i] * c[0];
    }
}
SMG_FN double kn_poly_value(const double* tab, int k, double t) {
    const double* c = tab + (size_t)(k < 0 ? 0 : (k >= kKnSteps ? kKnSteps - 1 : k)) * kKnStride;
    double p = c[kKnDeg];
#pragma unroll
    for (int j = kKnDeg - 1; j >= 0; --j) p = p * t + c[j];
    return p;
}
// Sum of n + 1 nodes from lo.
SMG_FN double kn_poly_sum(const double* tab, double lo, int n) {
    const double u = lo * (1.0 / kKnStep);
    const int k0 = (int)floor(u);
    const double t = u - (double)k0;
    const double a = kn_poly_value(tab, k0 + n, t);
    return k0 > 0 ? a - kn_poly_value(tab, k0 - 1, t) : a;
}

// Energy-window probability of a term with scattered energy ratio g = E'/E0
// (scatter.cu:1025-1033), FP64; erfc keeps the difference accurate when both
// ends lie on one side.
SMG_FN double window_prob(double e0, double lo, double hi, double res, double g) {
    const double ep = e0 * g, s2 = res * sqrt(g) / kFwhm * ep * sqrt(2.0);
    const double z1 = (lo - ep) / s2, z2 = (hi - ep) / s2;
    if (z1 >= 0.0) return 0.5 * (erfc(z1) - erfc(z2));
    if (z2 <= 0.0) return 0.5 * (erfc(-z2) - erfc(-z1));
    return 0.5 * (erf(z2) - erf(z1));
}

// The upper 2-sigma cut of a term (scatter.cu:1263-1269) rejects it when
// e0 g (1 - r sqrt(g)) >= hi, r = 2 res / FWHM; for r < 2/3 the left side grows
// with g on [0, 1], so the test is 1 - cos(theta) <= omc_hi for one value per
// row, found by bisection; -1 when nothing is rejected.
SMG_FN double window_reject_omc_hi(const ScatterPhys& ph) {
    const double alpha = ph.e0 / 511.0, r = ph.res * (2.0 / kFwhm);
    if (ph.e0 * (1.0 - r) < ph.hi) return -1.0;
    double g0 = 0.0, g1 = 1.0;  // below hi at g0, at or above it at g1
    for (int it = 0; it < 80; ++it) {
        const double gm = 0.5 * (g0 + g1);
        if (ph.e0 * gm * (1.0 - r * sqrt(gm)) >= ph.hi) g1 = gm;
        else g0 = gm;
    }
    return (1.0 / g1 - 1.0) / alpha;
}

// The window probability of a row as cubics over equal intervals of x =
// 1 - cos(theta), for the x the 2-sigma cuts leave: interval i holds 4 floats,
// value = ((c3 t + c2) t + c1) t + c0, t in [0, 1).  The probability is a Gaussian
// integral with its ends at z1, z2 standard deviations (times sqrt 2) from E':
// with z moving by at most kWinStep per interval the cubic through the interval's
// 4 Chebyshev points is within 2e-8 of it, relative.
constexpr double kWinStep = 0.04;
constexpr int kWinMin = 128, kWinMax = 1024;  // intervals

SMG_FN void win_cubic(const double v[4], float c[4]) {
    // Chebyshev points of [0, 1]
    const double x[4] = {0.5 * (1.0 - 0.92387953251128675613), 0.5 * (1.0 - 0.38268343236508977173),
                         0.5 * (1.0 + 0.38268343236508977173), 0.5 * (1.0 + 0.92387953251128675613)};
    double d[4] = {v[0], v[1], v[2], v[3]}, p[4] = {0.0, 0.0, 0.0, 0.0};
    for (int j = 1; j < 4; ++j)
        for (int i = 3; i >= j; --i) d[i] = (d[i] - d[i - 1]) / (x[i] - x[i - j]);
    for (int i = 3; i >= 0; --i) {
        for (int j = 3; j >= 1; --j) p[j] = p[j - 1] - x[i] * p[j];
        p[0] = d[i] - x[i] * p[0];
    }
    for (int i = 0; i < 4; ++i) c[i] = float(p[i]);
}
SMG_FN double win_point(int m) {
    return 0.5 * (1.0 + (m < 2 ? -1.0 : 1.0) * (m == 0 || m == 3 ? 0.92387953251128675613 : 0.38268343236508977173));
}
// Interval i of the table of a row with n intervals.
SMG_FN void win_interval(const ScatterPhys& ph, int i, float c[4]) {
    const double alpha = ph.e0 / 511.0;
    double v[4];
    for (int m = 0; m < 4; ++m) {
        const double x = ph.win_x0 + ((double)i + win_point(m)) / ph.win_scale;
        v[m] = window_prob(ph.e0, ph.lo, ph.hi, ph.res, 1.0 / (1.0 + alpha * x));
    }
    win_cubic(v, c);
}
// The table's domain from the row's cuts: cut is window_reject_cos(ph, 0).
SMG_FN void win_domain(ScatterPhys& ph, double cut, int n) {
    ph.omc_lo = cut < -1.5 ? 3.0 : (cut > 1.5 ? -1.0 : 1.0 - cut);
    ph.omc_hi = window_reject_omc_hi(ph);
    const double a = tmax2(ph.omc_hi, 0.0), b = tmin2(ph.omc_lo, 2.0);
    ph.win_n = n;
    ph.win_x0 = a;
    ph.win_scale = b > a ? (double)n / (b - a) : 1.0;
}
SMG_FN float win_table_value(const ScatterPhys& ph, double omc) {
    const double x = (omc - ph.win_x0) * ph.win_scale;
    int i = (int)x;
    i = i < 0 ? 0 : (i >= ph.win_n ? ph.win_n - 1 : i);
    const float t = float(x - (double)i);
    const float* c = ph.win + 4 * i;
    return ((c[3] * t + c[2]) * t + c[1]) * t + c[0];
}
// Intervals a row needs for kWinStep, or 0 when kWinMax do not do or the upper cut
// is not monotonic (a resolution above 78%): the FP32 term then evaluates the
// probability directly.  The bound takes the steepest slope of z over the whole
// domain, so what does not do depends on the window's width too: a window of +-10%
// has a table from 1% resolution up, 140.5 keV with 90-160 keV from 8%, 511 keV
// with 350-650 keV from 5%, 511 keV with 250-650 keV at none.
inline int win_intervals(const ScatterPhys& ph, double cut) {
    if (!(ph.res * (2.0 / kFwhm) < 0.66) || !(ph.res > 0.0) || !(ph.e0 > 0.0)) return 0;
    ScatterPhys q = ph;
    win_domain(q, cut, 1);
    const double alpha = q.e0 / 511.0, a = q.win_x0, b = a + 1.0 / q.win_scale;
    if (!(b > a)) return kWinMin;
    // |dz/dx| <= (|dE'/dx| / sigma + |lo or hi - E'| |dsigma/dx| / sigma^2) / sqrt 2,
    // largest at the interval's ends in g; bounded with the smallest sigma, and an
    // end of the window more than 7.5 sigma off (|z| > 5.3) is as good as infinite
    const double g0 = 1.0 / (1.0 + alpha * b), g1 = 1.0 / (1.0 + alpha * a);
    const double sig = q.res / kFwhm * q.e0 * g0 * sqrt(g0);
    const double far = tmin2(tmax2(tmax2(tabs(q.lo - q.e0 * g0), tabs(q.hi - q.e0 * g0)),
                                   tmax2(tabs(q.lo - q.e0 * g1), tabs(q.hi - q.e0 * g1))),
                             7.5 * q.res / kFwhm * q.e0 * g1 * sqrt(g1));
    const double dz = (q.e0 * alpha * g1 * g1 / sig + far * 1.5 * alpha * g1 / sig) / 1.4142135623730951;
    const double need = dz * (b - a) / kWinStep;
    for (int n = kWinMin; n <= kWinMax; n *= 2)
        if (need <= n) return n;
    return 0;
}

// Intervals of a launch with rows of resolutions res_lo to res_hi (ph: the window,
// or with same = false each row's own, E0 (1 -+ res / 2)): the largest need, which
// is not monotonic in the resolution (per-bar windows at 140.5 keV: 128 at 10% and
// 77%, 256 at 30%), over steps of at most 2; 0 when one of them has no table.
inline int win_intervals_rows(ScatterPhys ph, bool same, double res_lo, double res_hi) {
    const auto need = [&](double res) {
        ph.res = res;
        if (!same) {
            ph.lo = (1 - res / 2.0) * ph.e0;
            ph.hi = (1 + res / 2.0) * ph.e0;
        }
        return win_intervals(ph, window_reject_cos(ph, 0.0));
    };
    int n = need(res_lo);
    if (n == 0 || !(res_hi > res_lo)) return n;
    const int steps = (int)std::ceil(std::log(res_hi / res_lo) / std::log(2.0));
    for (int i = steps; i > 0; --i) {  // from the other end
        const int k = need(i == steps ? res_hi : res_lo * std::pow(res_hi / res_lo, (double)i / steps));
        if (k == 0) return 0;
        n = k > n ? k : n;
    }
    return n;
}

// atan2(s, c) for s >= 0, in [0, pi]: the smaller over the larger of s and |c|
// through a minimax polynomial of atan(a) / a in a^2 on [0, 1] (relative error
// 1.5e-8, fitted by Remez exchange), so a small angle keeps its relative precision.
SMG_FN float angle_f(float s, float c) {
    const float ac = tabs(c), hi = tmax2(s, ac), lo = tmin2(s, ac);
    const float a = hi > 0.0f ? lo * trcp(hi) : 0.0f, z = a * a;
    float p = 2.849889686e-03f;
    p = p * z - 1.606862992e-02f;
    p = p * z + 4.269152135e-02f;
    p = p * z - 7.504294813e-02f;
    p = p * z + 1.064093411e-01f;
    p = p * z - 1.420364380e-01f;
    p = p * z + 1.999261975e-01f;
    p = p * z - 3.333307207e-01f;
    p = p * z + 1.0f;
    float r = a * p;
    r = s > ac ? 1.57079632679489662f - r : r;
    return c < 0.0f ? 3.14159265358979324f - r : r;
}

// Per (scatter point, sub-cell) quantities shared by the lanes.
struct ScatterCell {
    double qs[3];        // scatter point, world
    double qss[3];       // scatter point, frame of bar d
    double q[3];         // sub-cell centre, world
    double lo[3], hi[3]; // sub-cell box, frame of bar d; corner c has lo[k] or hi[k]
                         // on axis k as bit k of c is clear or set
    PairTerm pt;
    const double* ic = nullptr;  // inv_corner of the 8 corners (PairRec), or formed per term
};

// True when the term of voxel p, scatter point sc.qs and sub-cell centre sc.q
// lies below the energy window by the per-row cosine threshold ph.c_rej
// (window_reject_cos): FP32 a.b < c_rej |a| |b|, or the FP64 cosine below
// it.  Such a term is 0 (scatter_term rejects it too); callers use this to
// skip the term, and loading its weight, early.
template <class T>
SMG_FN bool below_window(const ScatterPhys& ph, const double p[3], const ScatterCell& sc) {
    double a[3], b[3];
    for (int k = 0; k < 3; ++k) {
        a[k] = sc.qs[k] - p[k];
        b[k] = sc.q[k] - sc.qs[k];
    }
    if constexpr (std::is_same<T, float>::value) {
        const float ax = float(a[0]), ay = float(a[1]), az = float(a[2]);
        const float bx = float(b[0]), by = float(b[1]), bz = float(b[2]);
        const float ab = ax * bx + ay * by + az * bz;
        const float nn = (ax * ax + ay * ay + az * az) * (bx * bx + by * by + bz * bz);
        return ab < float(ph.c_rej) * tsqrt(nn);
    } else {
        const double dot = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
        const double na2 = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
        const double nb2 = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
        return dot / (sqrt(na2) * sqrt(nb2)) < ph.c_rej;
    }
}

// One (voxel, scatter point, sub-cell) term.  wgt is the weight of the
// scatter point for this voxel.  Returns 0 for terms outside the 2-sigma
// energy window (scatter.cu:1263-1269).  kTab: with the kernels' KN prefix
// polynomials, the FP32 pre-test of the window made by the caller; kWin (FP32):
// the row's window probability from its table, else evaluated here.
template <class T, bool kTab = false, bool kWin = kTab && std::is_same<T, float>::value>
SMG_FN T scatter_term(const ScatterPhys& ph, const double p[3], const double ps[3],
                      const ScatterCell& sc, T wgt, bool& near) {
    // Cone angle at the scatter point (scatter.cu:1254), scattered energy
    // (scatter.cu:1016-1023) and energy-window probability (scatter.cu:1025-1033).
    // The window probability sits on the tail of a Gaussian in E', which
    // multiplies the relative error of E' by ~50: E' and the window arguments
    // are formed in FP64 on both paths.  The FP64 path follows the reference
    // (acos of the clamped cosine, then cos of the angle); the fast path takes
    // cos and sin of the angle straight from the vectors.
    double a[3], b[3];
    for (int k = 0; k < 3; ++k) {
        a[k] = sc.qs[k] - p[k];
        b[k] = sc.q[k] - sc.qs[k];
    }
    if constexpr (std::is_same<T, float>::value) {
        // FP32 pre-test of the lower window cut (most terms of a scatter
        // matrix fall below the window): cos theta < c_rej  <=>
        // a.b < c_rej |a| |b|; a term near the cut goes on to the FP64 test
        // (kTab: the caller has made it)
        if constexpr (!kTab) {
            const float ax = float(a[0]), ay = float(a[1]), az = float(a[2]);
            const float bx = float(b[0]), by = float(b[1]), bz = float(b[2]);
            const float ab = ax * bx + ay * by + az * bz;
            const float nn = (ax * ax + ay * ay + az * az) * (bx * bx + by * by + bz * bz);
            if (ab < float(ph.c_rej) * tsqrt(nn)) return T(0);
        }
        // mu(E) tables without an FP32 form (more segments in range than it
        // holds): the whole term goes to the FP64 path, which keeps FP64
        // logarithms and exponentials out of the FP32 term
        if (ph.tab && ph.tab->n > 0 && !(ph.tabf && ph.tabf->n > 0)) {
            near = true;
            return T(0);
        }
    }
    const double alpha = ph.e0 / 511.0;
    double omc, st;  // 1 - cos(theta), sin(theta)
    {
        double dot = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
        double na2 = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
        double nb2 = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
        if constexpr (std::is_same<T, double>::value) {
            double c = dot / (sqrt(na2) * sqrt(nb2));
            if (c < ph.c_rej) return T(0);  // below the window (the test further down)
            if (c > 1.0) c = 1.0;
            if (c < -1.0) c = -1.0;
            omc = 1.0 - c;  // the reference's cos and sin of acos(c)
            st = sqrt((1.0 - c) * (1.0 + c));
        } else {
            // 1 - c and 1 - c^2 in FP64 keep nine digits at 0.001 rad
            const double c = tmax2(tmin2(dot * rsq_fast(na2 * nb2), 1.0), -1.0);
            omc = 1.0 - c;
            const double s2 = omc * (1.0 + c);
            st = s2 > 1e-300 ? s2 * rsq_fast(s2) : 0.0;
        }
    }
    // E' = E0 g with g = 1 / (1 + alpha (1 - cos)); the FP32 path forms the
    // window from g and one reciprocal, the FP64 path as the reference does
    double ep = 0.0, resp, z1 = 0.0, z2 = 0.0;
    T pe_win;
    if constexpr (kWin) {
        if (omc >= ph.omc_lo || omc <= ph.omc_hi) return T(0);  // scatter.cu:1263-1269
        pe_win = win_table_value(ph, omc);
    } else {
    if constexpr (std::is_same<T, double>::value) {
        ep = ph.e0 / (1.0 + alpha * omc);
        resp = ph.res * sqrt(ep / ph.e0);
        if (ep * (1 + 2 * resp / kFwhm) <= ph.lo || ep * (1 - 2 * resp / kFwhm) >= ph.hi)
            return T(0);  // 2-sigma energy-window early out (scatter.cu:1263-1269)
        double sigma = resp / kFwhm * ep;
        double s2 = sigma * sqrt(2.0);
        z1 = (ph.lo - ep) / s2;
        z2 = (ph.hi - ep) / s2;
    } else {
        // sigma sqrt(2) = resp E' sqrt(2) / FWHM
        constexpr double k2 = 2.0 / kFwhm, ks2 = 1.4142135623730950488 / kFwhm;
        const double g = rcp_fast(1.0 + alpha * omc);
        ep = ph.e0 * g;
        resp = ph.res * g * rsq_fast(g);
        if (ep * (1 + resp * k2) <= ph.lo || ep * (1 - resp * k2) >= ph.hi)
            return T(0);  // 2-sigma energy-window early out (scatter.cu:1263-1269)
        const double inv_s2 = resp > 0.0 ? rcp_fast(resp * ks2 * ep) : INFINITY;  // 1 / (sigma sqrt 2)
        z1 = (ph.lo - ep) * inv_s2;
        z2 = (ph.hi - ep) * inv_s2;
    }
    if constexpr (std::is_same<T, double>::value) {
        pe_win = 0.5 * (erf(z2) - erf(z1));
    } else {  // erfc keeps the difference accurate when both z lie on one side
        float f1 = float(z1), f2 = float(z2);
        if (z1 >= 0.0)
            pe_win = 0.5f * (erfcf(f1) - erfcf(f2));
        else if (z2 <= 0.0)
            pe_win = 0.5f * (erfcf(-f2) - erfcf(-f1));
        else
            pe_win = 0.5f * (erff(f2) - erff(f1));
    }
    }

    // azimuthal range from the sub-cell's bounding sphere (scatter.cu:1275-1287);
    // asin is ill-conditioned next to 1, where 1 - r is formed in FP64
    T phi;
    {
        const double L = sc.pt.len, rdet = ph.rcell;
        if (L * st * 2.0 <= rdet) {
            phi = T(kTwoPi);
        } else if constexpr (std::is_same<T, double>::value) {
            const double r = rdet / 2.0 / L / st;
            phi = 4.0 * asin(r <= 1.0 ? r : 1.0);
        } else {  // asin(r) as the angle of (r, sqrt((1 - r)(1 + r)))
            const double r = rdet * rcp_fast(2.0 * L * st);
            phi = 4.0f * angle_f(float(r), tsqrt(float(tmax2((1.0 - r) * (1.0 + r), 0.0))));
        }
    }
    const T alpha_t = T(alpha);

    // polar range: cone angles to the 8 sub-cell corners (scatter.cu:1290-1335).
    // The angle falls as its cosine grows, so the extreme cosines give the
    // extreme angles: no angle per corner (8 cross products and orderings per term
    // took the 1 mm collimator grid 354 ms instead of 323, the crystal grid 24.6
    // instead of 22.5).  The cosines are FP64 on both paths;
    // sin^2 = (1 - c)(1 + c) keeps a small angle's relative precision.
    T us[3];
    T tmin, tmax;
    double cmin = 0.0, cmax = 0.0;  // their cosines
    {
        double u[3], pl[3], ph8[3];
        for (int k = 0; k < 3; ++k) {
            u[k] = sc.qss[k] - ps[k];
            us[k] = T(u[k]);
            pl[k] = u[k] * (sc.lo[k] - sc.qss[k]);
            ph8[k] = u[k] * (sc.hi[k] - sc.qss[k]);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const double dot = ((c & 1 ? ph8[0] : pl[0]) + (c & 2 ? ph8[1] : pl[1])) + (c & 4 ? ph8[2] : pl[2]);
            const double cc = dot * (sc.ic ? sc.ic[c] : inv_corner(sc.lo, sc.hi, sc.qss, c));
            cmin = c == 0 ? cc : tmin2(cmin, cc);
            cmax = c == 0 ? cc : tmax2(cmax, cc);
        }
        const double u2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
        const double iu = std::is_same<T, double>::value ? 1.0 / sqrt(u2) : rsq_fast(u2);
        cmin = tmax2(tmin2(cmin * iu, 1.0), -1.0);
        cmax = tmax2(tmin2(cmax * iu, 1.0), -1.0);
        if constexpr (std::is_same<T, double>::value) {
            tmin = acos(cmax);
            tmax = acos(cmin);
        } else {
            tmin = angle_f(tsqrt(float((1.0 - cmax) * (1.0 + cmax))), float(cmax));
            tmax = angle_f(tsqrt(float((1.0 - cmin) * (1.0 + cmin))), float(cmin));
        }
    }
    // the line voxel -> scatter point, extended 1000 mm, through the sub-cell:
    // only the test of its chord against 0.001 is used.  FP32 path: a line that
    // passes the sub-cell's centre farther than its bounding radius + 0.01 mm has
    // chord 0 in the reference too (its small-component branches move the
    // line by less than 0.001 mm), so the chord is formed only otherwise.
    T lthru = T(0);
    bool lthru_needed = true;
    if constexpr (std::is_same<T, float>::value) {
        float w[3];
        for (int k = 0; k < 3; ++k) w[k] = float(0.5 * (sc.lo[k] + sc.hi[k]) - sc.qss[k]);
        const float cx = w[1] * us[2] - w[2] * us[1], cy = w[2] * us[0] - w[0] * us[2],
                    cz = w[0] * us[1] - w[1] * us[0];
        const float u2 = us[0] * us[0] + us[1] * us[1] + us[2] * us[2];
        const float R = float(ph.rcell) + 0.01f;
        lthru_needed = !(cx * cx + cy * cy + cz * cz > R * R * u2);
    }
    if (lthru_needed) {
        double D[3], dis2 = 0.0;
        for (int k = 0; k < 3; ++k) {
            D[k] = sc.qss[k] - ps[k];
            dis2 += D[k] * D[k];
        }
        if constexpr (std::is_same<T, float>::value) {
            // FP64 slab test of the extended line (length_box_ray; a line with one
            // component below eps must start strictly between that axis' faces
            // and runs over the other two, PESysMatGen.cu:69-73, and one with more
            // goes to the FP64 path): an FP32 form with tolerances on every
            // comparison takes three times the instructions.  The extension
            // leaves len / D_k as it is.
            const double idis = rsq_fast(dis2), dis = dis2 * idis, f = 1.0 + 1000.0 * idis;
            const double eps = kSlabEps<double>;
            double t0 = -1e300, t1 = 1e300;
            int ns = 0;
            bool in = true;
            for (int k = 0; k < 3; ++k) {
                const bool small = tabs(D[k] * f) < eps;
                const double inv = dis * rcp_fast(small ? 1.0 : D[k]);
                const double u = (sc.lo[k] - ps[k]) * inv, w = (sc.hi[k] - ps[k]) * inv;
                t0 = small ? t0 : tmax2(t0, tmin2(u, w));
                t1 = small ? t1 : tmin2(t1, tmax2(u, w));
                in = in && (!small || (ps[k] > sc.lo[k] && ps[k] < sc.hi[k]));
                ns += small;
            }
            near |= ns > 1;
            const double end = dis + 1000.0;
            const bool hit = in && t1 - t0 >= eps && t0 > eps && t1 < end;
            lthru = hit && t1 - t0 > (double)0.001f ? 1.0f : 0.0f;
        } else {
            const double dis = sqrt(dis2);
            double De[3];
            for (int k = 0; k < 3; ++k) De[k] = (sc.qss[k] + 1000.0 * D[k] / dis) - ps[k];
            SegDir<double> se;
            segdir_init<double>(se, De[0], De[1], De[2], 0.0, near);
            lthru = seg_box<double>(se, ps, sc.lo, sc.hi, near);
        }
    }
    if (lthru > T(0.001f)) tmin = T(0);
    T K;
    if constexpr (kTab) {
        int n;  // as the node loop forms it
        if constexpr (std::is_same<T, float>::value) {
            // a node count within the angles' rounding (below 1e-4 steps) of an
            // integer is formed from FP64 angles; sending the whole term to
            // FP64 for it (4 in 10,000 terms, so one in 40 of the 64 that a wave
            // evaluates together) took the 1 mm collimator grid 272 ms instead
            // of 263
            const float x = (tmax - tmin) * float(1.0 / kKnStep);
            n = (int)x;
            const float fr = x - float(n);
            if ((fr < 2e-4f && n > 0) || fr > 1.0f - 2e-4f)
                n = (int)((acos(cmin) - (tmin == 0.0f ? 0.0 : acos(cmax))) / kKnStep);
        } else {
            n = (int)((tmax - tmin) / kKnStep);
        }
        K = T(kn_poly_sum(ph.knp, double(tmin), n) * ph.inv_norm);
    } else if constexpr (std::is_same<T, double>::value)
        K = kn_sum<T>(tmin, tmax, alpha_t, near) / T(ph.norm);
    else if (ph.knt)
        K = float(kn_sum_table(ph.knt, tmin, tmax, near) / ph.norm);
    else
        K = kn_sum<T>(tmin, tmax, alpha_t, near) * float(1.0 / ph.norm);

    // second leg and absorption at E' (scatter.cu:1371-1427); the FP32 path
    // takes E0/E' = 1 + alpha (1 - cos) for the power laws
    // (FP32: tables here always have their FP32 form, see the entry test)
    double e3, e1;
    const bool tables = ph.tab && ph.tab->n > 0;
    float Lf = 0.0f;
    int jf = 0;
    if constexpr (std::is_same<T, float>::value) {
        if (!tables) {
            e1 = 1.0 + alpha * omc;
            e3 = e1 * e1 * e1;
        } else {
            Lf = log_f(float(1.0 + alpha * omc));  // ln(E0/E')
            jf = mu_seg_f(*ph.tabf, Lf);
            e3 = mu_ratio_f(*ph.tabf, 0, jf, Lf);
            e1 = mu_ratio_f(*ph.tabf, 1, jf, Lf);
        }
    } else {
        mu_ratios(ph.tab, ph.e0, ep, e3, e1);
    }
    double att2 = e3 * sc.pt.s_pe + e1 * sc.pt.s_c;
    if (sc.pt.s_wpe != 0.0 || sc.pt.s_wc != 0.0) {  // collimator material (grid scatterers)
        double w3 = e3, w1 = e1;
        if (tables) {
            if constexpr (std::is_same<T, float>::value) {
                w3 = mu_ratio_f(*ph.tabf, 2, jf, Lf);
                w1 = mu_ratio_f(*ph.tabf, 3, jf, Lf);
            } else {
                const double le = log(ep);
                w3 = exp(mu_table_log(*ph.tab, 2, le) - ph.tab->lmu0[2]);
                w1 = exp(mu_table_log(*ph.tab, 3, le) - ph.tab->lmu0[3]);
            }
        }
        att2 += w3 * sc.pt.s_wpe + w1 * sc.pt.s_wc;
    }
    double mupe = ph.mupe * e3;
    double mut = mupe + ph.muc * e1;
    T ea = exp_neg<T>(sc.pt.la * mut);
    if constexpr (std::is_same<T, double>::value) {
        T absf = (T(1) - ea) * T(mupe / mut);
        return wgt * phi / T(kTwoPi) * K * pe_win * exp_neg<T>(att2) * absf;
    } else {
        T absf = (T(1) - ea) * tdiv(float(mupe), float(mut));
        return wgt * phi * float(1.0 / kTwoPi) * K * pe_win * exp_neg<T>(att2) * absf;
    }
}

}  // namespace smg
