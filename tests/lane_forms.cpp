// Host build of the scatter terms as the kernels form them (KN prefix polynomials,
// reciprocal corner distances, and in FP32 the window probability from the row's
// table or evaluated per term), for tests/test_scatter_forms.py.
#include "lane_harness.cpp"

namespace {

std::vector<double> kn_polys(double e0) {
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
    return tab;
}

template <class T, bool kWin>
double form_element(const Ctx& c, const double* knp, const float* pe, const uint32_t* bitmap, int kind, int variant,
                    int d, int v, int rot, const int sub[3], long* fallbacks) {
    const PeGeom& G = c.G;
    const GeomDesc& g = G.g;
    const Bar<double>& bd = G.bars_d[d];
    const float* ph = c.hg.phys.data();
    if (!(bd.mut > (double)0.01f)) return 0.0;
    const int nxy = g.nx * g.ny, rem = v % nxy;
    const double phi = (double)rot * g.dphi;
    double p[3], ps[3];
    voxel_position(g, rem % g.nx, rem / g.nx, v / nxy, std::cos(phi), std::sin(phi), p);
    to_frame(bd, p, ps);
    ScatterPhys P;
    P.e0 = ph[7];
    const bool same = (int)std::floor((double)ph[4] + 0.5) > 0;
    P.lo = same ? (double)ph[5] : (1 - bd.res / 2.0) * P.e0;
    P.hi = same ? (double)ph[6] : (1 + bd.res / 2.0) * P.e0;
    P.res = bd.res;
    P.norm = kn_norm(P.e0);
    P.inv_norm = 1.0 / P.norm;
    P.mupe = bd.mupe;
    P.muc = bd.muc;
    P.rcell = std::sqrt(bd.w * bd.w / sub[0] / sub[0] + bd.h * bd.h / sub[2] / sub[2] + bd.t * bd.t / sub[1] / sub[1]) / 2.0;
    P.knp = knp;
    const double cut = window_reject_cos(P, 0.0);
    P.c_rej = window_cut_margin(cut, std::is_same<T, double>::value ? 1e-9 : 1e-5);
    std::vector<float> win;
    if (kWin) {
        const int nw = win_intervals(P, cut);
        if (nw == 0) return -1.0;
        win_domain(P, cut, nw);
        win.resize((size_t)nw * 4);
        for (int i = 0; i < nw; ++i) win_interval(P, i, &win[4 * (size_t)i]);
        P.win = win.data();
    }
    KahanSum<T> acc;
    for (int cell = 0; cell < sub[0] * sub[1] * sub[2]; ++cell) {
        CellCtx cc;
        make_cell_ctx(bd, cell % sub[0], (cell / sub[0]) % sub[1], cell / (sub[0] * sub[1]), sub[0], sub[1], sub[2], cc);
        ScatterCell sc;
        for (int k = 0; k < 3; ++k) {
            sc.q[k] = cc.q[k];
            sc.lo[k] = cc.lo[k];
            sc.hi[k] = cc.hi[k];
        }
        for (int s = 0; s < (kind == 0 ? g.n_det : c.hg.n_holes_l0); ++s) {
            if (kind == 0 && s == d) continue;
            double dyh = 0.0;
            if (kind == 0) {
                const Bar<double>& bs = G.bars_d[s];
                sc.qs[0] = bs.cx;
                sc.qs[1] = bs.cy;
                sc.qs[2] = bs.cz;
            } else {
                const float* hp = c.hg.coll.data() + 100 + 9 * s;
                sc.qs[0] = hp[0];
                sc.qs[1] = ((double)hp[1] + (double)hp[2]) / 2.0 + g.fov2coll;
                sc.qs[2] = hp[3];
                dyh = (double)hp[2] - (double)hp[1];
            }
            to_frame(bd, sc.qs, sc.qss);
            if (std::is_same<T, float>::value && below_window<float>(P, p, sc)) continue;  // the kernel's pre-test
            sc.pt = pair_term(c, bitmap, kind, d, s, sc.qs, cc);
            double ic[8];
            for (int k = 0; k < 8; ++k) ic[k] = inv_corner(cc.lo, cc.hi, sc.qss, k);
            sc.ic = ic;
            T wgt;
            if (kind == 0) {
                wgt = T(pe[(int64_t)s * g.n_vox + v]) * T(bd.muc / bd.mupe);
            } else {
                const double dx = p[0] - sc.qs[0], dy = p[1] - sc.qs[1], dz = p[2] - sc.qs[2];
                const double lv = std::sqrt(dx * dx + dy * dy + dz * dz), r = variant == 0 ? (double)0.1f : (double)0.2f;
                const double om = variant == 0 ? (r * r * 3.14159265358979323846 + dyh * r) /
                                                     (4.0 * 3.14159265358979323846 * lv * lv) * std::fabs(dy) / lv
                                               : (r * r + dyh * r) / (4.0 * lv * lv);
                wgt = T(om * ((double)c.hg.coll[17] / (double)c.hg.coll[15]));
            }
            bool near = false;
            T val = scatter_term<T, true, kWin>(P, p, ps, sc, wgt, near);
            if (near) {
                bool n2 = false;
                val = T(scatter_term<double, true>(P, p, ps, sc, double(wgt), n2));
                ++*fallbacks;
            }
            acc.add(val);
        }
    }
    return (double)(float)acc.value();
}

}  // namespace

extern "C" {

// form 0: FP64; 1: FP32 with the row's window table (an element of -1: the row has
// none); 2: FP32 with the window probability per term.  Returns the FP64
// re-computations.
long form_scatter_pairs(const float* coll, const float* det, const float* img, const float* phys, const float* pe,
                        const uint32_t* bitmap, int kind, int variant, int rot, int sx, int sy, int sz, int form,
                        const int* d, const int* v, int n, double* out) {
    Ctx c;
    if (!make_ctx(coll, det, img, phys, c)) return -1;
    const std::vector<double> knp = kn_polys(phys[7]);
    const int sub[3] = {sx, sy, sz};
    long fb = 0;
    for (int i = 0; i < n; ++i) {
        if (form == 0)
            out[i] = form_element<double, false>(c, knp.data(), pe, bitmap, kind, variant, d[i], v[i], rot, sub, &fb);
        else if (form == 1)
            out[i] = form_element<float, true>(c, knp.data(), pe, bitmap, kind, variant, d[i], v[i], rot, sub, &fb);
        else
            out[i] = form_element<float, false>(c, knp.data(), pe, bitmap, kind, variant, d[i], v[i], rot, sub, &fb);
    }
    return fb;
}

}  // extern "C"

extern "C" {

// Intervals of the window tables: one row, and a launch with rows of resolutions
// res_lo to res_hi (same = 0: each row's own window).
int form_row_intervals(double e0, double lo, double hi, double res) {
    ScatterPhys P;
    P.e0 = e0;
    P.lo = lo;
    P.hi = hi;
    P.res = res;
    return win_intervals(P, window_reject_cos(P, 0.0));
}
int form_launch_intervals(double e0, double lo, double hi, int same, double res_lo, double res_hi) {
    ScatterPhys P;
    P.e0 = e0;
    P.lo = lo;
    P.hi = hi;
    return win_intervals_rows(P, same != 0, res_lo, res_hi);
}

}  // extern "C"
