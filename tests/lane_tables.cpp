// Host build of the scatter kernels' tables, for tests/test_lane_tables.py.
#include <cmath>
#include <vector>

#include "smg_scatter_body.hpp"

using namespace smg;

extern "C" {

// KN rectangle sums over [lo[i], hi[i]] from the prefix polynomials of e0.
void table_kn_sums(double e0, const double* lo, const double* hi, int n, double* out) {
    std::vector<double> tab((size_t)kKnPolySize, 0.0);
    std::vector<KahanSum<double>> acc(kKnDeg + 1);
    for (int k = 0; k < kKnSteps; ++k) {
        double v[kKnDeg + 1];
        for (int m = 0; m <= kKnDeg; ++m) {
            acc[m].add(kn_node(e0 / 511.0, kn_phase(m), k));
            v[m] = acc[m].value();
        }
        kn_poly_coeffs(v, &tab[(size_t)k * kKnStride]);
    }
    for (int i = 0; i < n; ++i) out[i] = kn_poly_sum(tab.data(), lo[i], (int)((hi[i] - lo[i]) / kKnStep));
}

// Window probability of a row at 1 - cos(theta) = omc[i] from its table (FP32)
// and directly; pass[i]: the 2-sigma cuts keep the term, by the table's limits
// and by the reference's tests.  Returns the table's intervals (0: none).
int table_window(double e0, double lo, double hi, double res, const double* omc, int n, double* tab_out,
                 double* direct, int* pass_tab, int* pass_ref) {
    ScatterPhys ph;
    ph.e0 = e0;
    ph.lo = lo;
    ph.hi = hi;
    ph.res = res;
    const double cut = window_reject_cos(ph, 0.0);
    const int nw = win_intervals(ph, cut);
    if (nw == 0) return 0;
    win_domain(ph, cut, nw);
    std::vector<float> tab((size_t)nw * 4);
    for (int i = 0; i < nw; ++i) win_interval(ph, i, &tab[4 * (size_t)i]);
    ph.win = tab.data();
    for (int i = 0; i < n; ++i) {
        const double g = 1.0 / (1.0 + e0 / 511.0 * omc[i]), ep = e0 * g, resp = res * std::sqrt(g);
        tab_out[i] = win_table_value(ph, omc[i]);
        direct[i] = window_prob(e0, lo, hi, res, g);
        pass_tab[i] = !(omc[i] >= ph.omc_lo || omc[i] <= ph.omc_hi);
        pass_ref[i] = !(ep * (1 + 2 * resp / kFwhm) <= lo || ep * (1 - 2 * resp / kFwhm) >= hi);
    }
    return nw;
}

void table_angles(const float* s, const float* c, int n, float* out) {
    for (int i = 0; i < n; ++i) out[i] = angle_f(s[i], c[i]);
}

}  // extern "C"
