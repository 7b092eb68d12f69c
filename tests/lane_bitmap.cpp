// Host build of the bitmap kernel's decisions, for tests/test_lane_bitmap.py.
#include <algorithm>

#include "smg_bitmap_body.hpp"

using namespace smg;

extern "C" {

// All (i, j, k), i < j, of n spheres (x, y, z, r).  The decisions that bm_margin
// takes by itself against the reference's test in FP64: wrong ones, the number left
// to FP64, and the largest error of a margin whose FP64 value is below 0.05.
void bitmap_decisions(const double* sph, int n, int coll, long* wrong, long* left, double* err) {
    const Sphere<double>* s = (const Sphere<double>*)sph;
    *wrong = *left = 0;
    *err = 0.0;
    for (int i = 0; i < n; ++i)
        for (int j = coll ? 0 : i + 1; j < n; ++j) {
            const BmRow r = bm_row(s[i], s[j]);
            for (int k = 0; k < n; ++k) {
                if (k == i || k == j) continue;
                float t = bm_margin(bm_dir(s[i], s[k]), r.x2, r.y2, r.z2, r.c);
                const double lij = bm_dist(s[i].x, s[i].y, s[i].z, s[j].x, s[j].y, s[j].z);
                const double lik = bm_dist(s[i].x, s[i].y, s[i].z, s[k].x, s[k].y, s[k].z);
                if (lij > 0 && lik > 0) {
                    const double ux = (s[k].x - s[i].x) / lik - (s[j].x - s[i].x) / lij;
                    const double uy = (s[k].y - s[i].y) / lik - (s[j].y - s[i].y) / lij;
                    const double uz = (s[k].z - s[i].z) / lik - (s[j].z - s[i].z) / lij;
                    const double lim = s[k].r / lik + s[j].r / lij, t64 = lim * lim - ux * ux - uy * uy - uz * uz;
                    if (std::abs(t64) < 0.05) *err = std::max(*err, std::abs(t - t64));
                }
                if (!coll) t = std::fmax(t, bm_margin(bm_dir(s[j], s[k]), -r.x2, -r.y2, -r.z2, r.cr));
                if (std::abs(t) <= kBmTol) {
                    ++*left;
                    continue;
                }
                bool nn = false;
                const bool want = coll ? bm_seen_from<double>(s[i], s[j], s[k], nn)
                                       : bm_crystal_pred<double>(s[i], s[j], s[k], nn);
                *wrong += (t > 0.0f) != want;
            }
        }
}

}  // extern "C"
