// Host build of the wave-level candidate tests of the PE kernels (tile box,
// sub-cell point), for tests/test_lane_tiles.py.
#include <algorithm>
#include <cstdint>
#include <string>
#include <vector>

#include "smg_parse.hpp"
#include "smg_pe_body.hpp"

using namespace smg;

extern "C" {

// n_waves seeded (bar, tile) pairs: every bar and hole whose reference chord
// (no culling) is above 0 for some lane's ray to some sub-cell must pass the
// tile test (bar_tile_may_hit) and the sub-cell test (box_meets_frustum) with
// the tile's extents.  stats[0] chords above 0, [1] of them dropped by the
// tile test, [2] by the sub-cell test, [3] (candidate, sub-cell) pairs kept
// with the extents, [4] with the bounding ball, [5] kept with the extents but
// not with the ball.
int tile_extent_check(const float* coll, const float* det, const float* img, const float* phys,
                      const float* shapes, int n_shapes, int rot, int sx, int sy, int sz, int tx, int ty,
                      int tz, int n_waves, unsigned seed, double* stats) {
    HostGeom hg;
    std::string why;
    if (parse_geometry(coll, det, img, phys, hg, why) != 0) return -1;
    if (n_shapes > 0 && apply_hole_shapes(hg, shapes, n_shapes, why) != 0) return -1;
    const GeomDesc& g = hg.g;
    const int tile[3] = {tx, ty, tz};
    const int nt[3] = {(g.nx + tx - 1) / tx, (g.ny + ty - 1) / ty, (g.nz + tz - 1) / tz};
    const double phi = (double)rot * g.dphi, cphi = std::cos(phi), sphi = std::sin(phi);
    uint64_t st = seed * 2654435761ull + 1;
    auto next = [&]() {
        st ^= st << 13;
        st ^= st >> 7;
        st ^= st << 17;
        return st;
    };
    for (int i = 0; i < 6; ++i) stats[i] = 0.0;
    for (int w = 0; w < n_waves; ++w) {
        const int d = (int)(next() % g.n_det);
        const int t = (int)(next() % ((uint64_t)nt[0] * nt[1] * nt[2]));
        const int ix0 = (t % nt[0]) * tx, iy0 = ((t / nt[0]) % nt[1]) * ty, iz0 = (t / (nt[0] * nt[1])) * tz;
        const Bar<double>& bd = hg.bars_d[d];
        const Bar<float>& bdf = hg.bars_f[d];
        double tc[3], rho;
        tile_ball(g, ix0, iy0, iz0, tile, cphi, sphi, tc, rho);
        float tcf[3], rhof, te[3];
        tile_ball_f(tc, rho, tcf, rhof);
        tile_extents(g, ix0, iy0, iz0, tile, cphi, sphi, te);
        const float rq[3] = {0.0f, 0.0f, 0.0f};
        for (int k = 0; k < g.n_det + g.n_holes; ++k) {
            if (k == d) continue;
            const bool is_bar = k < g.n_det;
            float c[3], cb = 1.0f, sb = 0.0f, h[3], rt[3];
            if (is_bar) {
                const Bar<float>& b = hg.bars_f[k];
                c[0] = b.cx; c[1] = b.cy; c[2] = b.cz;
                cb = b.cb; sb = b.sb;
                h[0] = 0.5f * b.w; h[1] = 0.5f * b.t; h[2] = 0.5f * b.h;
            } else {
                const Hole<float>& o = hg.holes_f[k - g.n_det];
                c[0] = o.xc; c[1] = o.ymid; c[2] = o.zc;
                h[0] = o.r; h[1] = 0.5f * tabs(o.y2 - o.y1); h[2] = o.r;
            }
            extents_in_frame(te, cb, sb, rt);
            const bool hit_tile = bar_tile_may_hit(bdf, tcf, rt, c[0], c[1], c[2], cb, sb, h[0], h[1], h[2]);
            for (int cell = 0; cell < sx * sy * sz; ++cell) {
                const int sub[3] = {sx, sy, sz};
                CellCtx cc;
                make_cell_ctx_linear(bd, cell, sub, cc);
                const float q[3] = {float(cc.q[0]), float(cc.q[1]), float(cc.q[2])};
                const bool hit_cell = box_meets_frustum(q, rq, tcf, rt, c[0], c[1], c[2], cb, sb, h[0], h[1], h[2]);
                const bool ball = box_meets_frustum(q, rq, tcf, rhof, c[0], c[1], c[2], cb, sb, h[0], h[1], h[2]);
                stats[3] += hit_cell;
                stats[4] += ball;
                stats[5] += hit_cell && !ball;
                for (int l = 0; l < tx * ty * tz; ++l) {
                    const int ix = ix0 + l % tx, iy = iy0 + (l / tx) % ty, iz = iz0 + l / (tx * ty);
                    if (ix >= g.nx || iy >= g.ny || iz >= g.nz) continue;
                    double p[3];
                    voxel_position(g, ix, iy, iz, cphi, sphi, p);
                    double D[3] = {cc.q[0] - p[0], cc.q[1] - p[1], cc.q[2] - p[2]};
                    double len = 0.0;
                    bool near = false;
                    if (is_bar) {
                        const Bar<double>& b = hg.bars_d[k];
                        double a[3], e[3];
                        to_frame(b, p, a);
                        to_frame(b, cc.q, e);
                        const double lo[3] = {-0.5 * b.w, -0.5 * b.t, -0.5 * b.h};
                        const double hi[3] = {0.5 * b.w, 0.5 * b.t, 0.5 * b.h};
                        SegDir<double> s;
                        segdir_init<double>(s, e[0] - a[0], e[1] - a[1], e[2] - a[2], 0.0, near);
                        len = seg_box<double>(s, a, lo, hi, near);
                    } else {
                        const Hole<double>& o = hg.holes_d[k - g.n_det];
                        const double dd = sqrt(D[0] * D[0] + D[1] * D[1] + D[2] * D[2]);
                        CylRay cr;
                        cyl_ray(D, dd, cr);
                        len = o.erx > 0.0 ? ell_chord(o, p[0], p[1], p[2], cr.kx, cr.kz, cr.inv_ky, dd)
                                          : cyl_chord(p, cr, dd, o.xc, o.y1, o.y2, o.zc, o.r);
                    }
                    if (!(len > 0.0)) continue;
                    stats[0] += 1;
                    stats[1] += !hit_tile;
                    stats[2] += !hit_cell;
                }
            }
        }
    }
    return 0;
}

// n_waves seeded (bar, tile) pairs: a bar or hole that cull_keeps_all keeps for
// the whole tile must pass the reference culling test (FP64) of every voxel of
// the tile.  stats[0] candidates kept for all, [1] of them failing some voxel's
// test, [2] candidates every voxel's test keeps.
int cull_all_check(const float* coll, const float* det, const float* img, const float* phys, int rot, int tx,
                   int ty, int tz, int n_waves, unsigned seed, double* stats) {
    HostGeom hg;
    std::string why;
    if (parse_geometry(coll, det, img, phys, hg, why) != 0) return -1;
    const GeomDesc& g = hg.g;
    PeGeom G{};
    G.g = g;
    G.bars_f = hg.bars_f.data();
    G.bars_d = hg.bars_d.data();
    G.holes_f = hg.holes_f.data();
    G.holes_d = hg.holes_d.data();
    const int tile[3] = {tx, ty, tz};
    const int nt[3] = {(g.nx + tx - 1) / tx, (g.ny + ty - 1) / ty, (g.nz + tz - 1) / tz};
    const double phi = (double)rot * g.dphi, cphi = std::cos(phi), sphi = std::sin(phi);
    uint64_t st = seed * 2654435761ull + 1;
    auto next = [&]() {
        st ^= st << 13;
        st ^= st >> 7;
        st ^= st << 17;
        return st;
    };
    for (int i = 0; i < 3; ++i) stats[i] = 0.0;
    for (int w = 0; w < n_waves; ++w) {
        const int d = (int)(next() % g.n_det);
        const int t = (int)(next() % ((uint64_t)nt[0] * nt[1] * nt[2]));
        const int ix0 = (t % nt[0]) * tx, iy0 = ((t / nt[0]) % nt[1]) * ty, iz0 = (t / (nt[0] * nt[1])) * tz;
        const Bar<float>& bdf = hg.bars_f[d];
        double tc[3], rho;
        tile_ball(g, ix0, iy0, iz0, tile, cphi, sphi, tc, rho);
        float tcf[3], rhof;
        tile_ball_f(tc, rho, tcf, rhof);
        const float cd[3] = {bdf.cx, bdf.cy, bdf.cz};
        for (int k = 0; k < g.n_det + g.n_holes; ++k) {
            if (k == d) continue;
            const bool is_bar = k < g.n_det;
            float c[3], num;
            if (is_bar) {
                const Bar<float>& b = hg.bars_f[k];
                c[0] = b.cx; c[1] = b.cy; c[2] = b.cz;
                num = 0.5f * b.rdiag;
            } else {
                const Hole<float>& o = hg.holes_f[k - g.n_det];
                c[0] = o.xc; c[1] = o.ymid; c[2] = o.zc;
                num = o.crit;
            }
            const bool all = cull_keeps_all(tcf, rhof, c, num, cd, 0.5f * bdf.rdiag);
            bool every = true;
            for (int l = 0; l < tx * ty * tz; ++l) {
                const int ix = ix0 + l % tx, iy = iy0 + (l / tx) % ty, iz = iz0 + l / (tx * ty);
                if (ix >= g.nx || iy >= g.ny || iz >= g.nz) continue;
                double p[3];
                voxel_position(g, ix, iy, iz, cphi, sphi, p);
                const float pf[3] = {float(p[0]), float(p[1]), float(p[2])}, udf[3] = {0, 0, 0};
                SelfCull sc;
                self_cull(hg.bars_d[d], p, sc);
                every &= is_bar ? cull_bar<true>(G, k, p, pf, sc, udf, 0.0f)
                                : cull_hole<true>(G, k - g.n_det, p, pf, sc, udf, 0.0f);
            }
            stats[0] += all;
            stats[1] += all && !every;
            stats[2] += every;
        }
    }
    return 0;
}

}  // extern "C"
