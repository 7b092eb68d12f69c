// Primary-Compton scatter matrices for gfx950: crystal scatter (scatter point
// = centre of another bar, weighted by the PE matrix) and collimator scatter
// (scatter point = centre of a layer-0 hole, weighted by a virtual-disc solid
// angle).  References: ScatterGen_RayTracing_CircularHole/scatter.cu:1077-1437
// and :1544-1936, ScatterGen_Collimator/scatter.cu:1056-1435.
//
// Two kernels:
//   pair_terms_kernel  one record per (bar d, scatter point s, sub-cell): the
//                      voxel-independent second-leg sums S_pe, S_c over the
//                      bars flagged in the geometry bitmap, the own-bar path
//                      and the absorption chord, in FP64.
//   scatter_kernel     one wave per (bar d, 64 consecutive voxels[, slice of
//                      the scatter points]); each lane owns one element and
//                      loops over scatter points and sub-cells, summing with
//                      a two-sum compensated sum.  When the points are split
//                      into slices, scatter_reduce_kernel adds the slices'
//                      sums in slice order.
//                      The reference instead runs one thread per
//                      (d, v, s) and sums with float atomicAdd, in an order
//                      that changes from run to run (scatter.cu:1427).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "smg_kernels.hpp"
#include "smg_scatter_body.hpp"

namespace smg {

namespace {

// The bar of output row r.
__device__ __forceinline__ int row_bar(const ScatterLaunch& A, int r) { return A.rows ? A.rows[r] : A.row0 + r; }

// The energy window of bar d's row.
__device__ __forceinline__ void row_phys(const ScatterLaunch& A, const Bar<double>& bd, ScatterPhys& ph) {
    ph.e0 = A.e0;
    if (A.same_window) {
        ph.lo = A.win_lo;
        ph.hi = A.win_hi;
    } else {  // per-bar window E0 (1 -+ res/2) (scatter.cu:1154-1163)
        ph.lo = (1 - bd.res / 2.0) * A.e0;
        ph.hi = (1 + bd.res / 2.0) * A.e0;
    }
    ph.res = bd.res;
}

// One thread per output row: its energy-window cut (window_reject_cos with no
// margin), and the domain of its window table, once per launch instead of once
// per pair-term thread and per scatter wave (80-step FP64 bisections).
__global__ __launch_bounds__(64) void row_cut_kernel(ScatterLaunch A, double* cut, WinRow* win) {
    const int r = (int)(blockIdx.x * 64 + threadIdx.x);
    if (r >= A.n_rows) return;
    ScatterPhys ph;
    row_phys(A, A.geom.bars_d[row_bar(A, r)], ph);
    cut[r] = window_reject_cos(ph, 0.0);
    if (A.win_n > 0) {
        win_domain(ph, cut[r], A.win_n);
        win[r] = WinRow{ph.win_x0, ph.win_scale, ph.omc_lo, ph.omc_hi};
    }
}

// One thread per interval of a row's window table.
__global__ __launch_bounds__(256) void win_table_kernel(ScatterLaunch A, const WinRow* win, float* tab) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= (int64_t)A.n_rows * A.win_n) return;
    const int r = (int)(tid / A.win_n), i = (int)(tid % A.win_n);
    ScatterPhys ph;
    row_phys(A, A.geom.bars_d[row_bar(A, r)], ph);
    ph.win_x0 = win[r].x0;
    ph.win_scale = win[r].scale;
    float c[4];
    win_interval(ph, i, c);
    *(float4*)(tab + 4 * tid) = make_float4(c[0], c[1], c[2], c[3]);
}

// True when the terms of scatter point qs and sub-cell centre q lie below the
// energy window for every voxel of the image, so scatter_kernel's per-lane
// test (below_window, cosine threshold c_lo - 1e-5 in FP32, c_lo - 1e-9 in
// FP64) rejects each of them before it reads the pair term; c_lo is the row's
// cut (row_window_cos).  The voxel centres lie in a ball (C, R); seen from qs
// they are within asin(R / |qs - C|) of the direction qs - C, so no voxel's
// cosine exceeds cos(angle(qs - C, q - qs) - asin(R / |qs - C|)); the test
// asks that bound to be 1e-4 below the FP32 threshold.
__device__ bool below_window_all(const ScatterLaunch& A, double c_lo, const double qs[3],
                                 const double q[3]) {
    if (c_lo <= -1.5) return false;  // nothing is rejected
    const GeomDesc& g = A.geom.g;
    const int whole[3] = {g.nx, g.ny, g.nz};
    double C[3], R;
    tile_ball(g, 0, 0, 0, whole, A.cphi, A.sphi, C, R);
    double u[3], b[3];
    for (int k = 0; k < 3; ++k) {
        u[k] = qs[k] - C[k];
        b[k] = q[k] - qs[k];
    }
    const double L = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double B = sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
    if (!(L > R * (1.0 + 1e-9) + 1e-9) || !(B > 0.0)) return false;
    double cu = (u[0] * b[0] + u[1] * b[1] + u[2] * b[2]) / (L * B);
    cu = cu > 1.0 ? 1.0 : (cu < -1.0 ? -1.0 : cu);
    const double th = acos(cu) - asin(R / L);
    if (!(th > 0.0)) return false;
    return cos(th) < c_lo - 1.1e-4;
}

__device__ __forceinline__ double readlane_d(double x, int lane) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// One (row, scatter point, sub-cell) record: its indices and points.
struct PairIds {
    int r, s, d, sbar;
    CellCtx cc;
    double qs[3];
};
__device__ __forceinline__ void pair_ids(const ScatterLaunch& A, int64_t tid, PairIds& P) {
    const int ncell = A.sub[0] * A.sub[1] * A.sub[2];
    const int cell = (int)(tid % ncell);
    P.s = (int)((tid / ncell) % A.n_pts);
    P.r = (int)(tid / ((int64_t)ncell * A.n_pts));
    P.d = row_bar(A, P.r);
    // the bar holding the scatter point (crystal scatter)
    P.sbar = A.kind == 3 ? A.pt_bar0 + P.s / A.pts_per_bar : P.s;
    const int a = cell % A.sub[0], b = (cell / A.sub[0]) % A.sub[1], c = cell / (A.sub[0] * A.sub[1]);
    make_cell_ctx(A.geom.bars_d[P.d], a, b, c, A.sub[0], A.sub[1], A.sub[2], P.cc);
    const ScatterPt<double>& sp = A.pts_d[P.s];
    P.qs[0] = sp.x;
    P.qs[1] = sp.y;
    P.qs[2] = sp.z;
}

// Chord of the second leg qs -> q through bar k.  In the frame of an unturned
// bar (beta = 0) the segment's direction is q - qs, the same for every such bar:
// its direction data (length, the eps decisions, len / D_k) are formed once per
// record, in sdw.  A turned bar gets its own.
__device__ __forceinline__ double leg_chord(const Bar<double>& bk, const SegDir<double>& sdw, const double qs[3],
                                            const double q[3]) {
    bool near = false;
    const double lo[3] = {-0.5 * bk.w, -0.5 * bk.t, -0.5 * bk.h};
    const double hi[3] = {0.5 * bk.w, 0.5 * bk.t, 0.5 * bk.h};
    if (bk.sb == 0.0 && bk.cb == 1.0) {
        const double pa[3] = {qs[0] - bk.cx, qs[1] - bk.cy, qs[2] - bk.cz};
        return seg_box<double>(sdw, pa, lo, hi, near);
    }
    double pa[3], pb[3];
    to_frame(bk, qs, pa);
    to_frame(bk, q, pb);
    SegDir<double> sd;
    segdir_init<double>(sd, pb[0] - pa[0], pb[1] - pa[1], pb[2] - pa[2], 0.0, near);
    return seg_box<double>(sd, pa, lo, hi, near);
}

// The rest of a record after the other bars' sums in out, and its store.
__device__ __forceinline__ void finish_pair(const ScatterLaunch& A, const PairIds& P, PairTerm& out, PairRec& rec) {
    const PeGeom& G = A.geom;
    const Bar<double>& bd = G.bars_d[P.d];
    const CellCtx& cc = P.cc;
    bool near = false;
    if (A.kind == 2) {  // collimator material from the grid point to the sub-cell
        double att_t;
        coll_material(G, P.qs, cc.q, att_t, out.s_wpe, out.s_wc);
    }
    if (A.kind == 3) {  // grid point inside bar sbar: its way out of that bar
        const Bar<double>& bs = G.bars_d[P.sbar];
        double sa[3], qa[3];
        to_frame(bs, P.qs, sa);
        to_frame(bs, cc.q, qa);
        const double lo[3] = {-0.5 * bs.w, -0.5 * bs.t, -0.5 * bs.h};
        const double hi[3] = {0.5 * bs.w, 0.5 * bs.t, 0.5 * bs.h};
        const double l = seg_box_geo(sa, qa, lo, hi);
        out.s_pe += l * bs.mupe;
        out.s_c += l * bs.muc;
    }
    // own bar from its surface to the sub-cell (scatter.cu:1405-1417)
    double qss[3];
    to_frame(bd, P.qs, qss);
    double blo[3] = {-bd.w / 2.0, -bd.t / 2.0, -bd.h / 2.0};
    double bhi[3] = {bd.w / 2.0, bd.t / 2.0, bd.h / 2.0};
    SegDir<double> so;
    segdir_init<double>(so, cc.qs[0] - qss[0], cc.qs[1] - qss[1], cc.qs[2] - qss[2], 0.0, near);
    double l1 = seg_box_inside<double>(so, qss, blo, bhi, near);
    double l2 = seg_box_inside<double>(so, qss, cc.lo, cc.hi, near);
    out.s_pe += (l1 - l2) * bd.mupe;
    out.s_c += (l1 - l2) * bd.muc;
    // absorption chord, ray extended 1000 mm through the sub-cell (scatter.cu:1420-1424)
    double dx = P.qs[0] - cc.q[0], dy = P.qs[1] - cc.q[1], dz = P.qs[2] - cc.q[2];
    out.len = sqrt(dx * dx + dy * dy + dz * dz);
    double De[3];
    for (int k = 0; k < 3; ++k) De[k] = (cc.qs[k] + 1000.0 * (cc.qs[k] - qss[k]) / out.len) - qss[k];
    SegDir<double> se;
    segdir_init<double>(se, De[0], De[1], De[2], 0.0, near);
    out.la = seg_box<double>(se, qss, cc.lo, cc.hi, near);
    rec.t = out;
    for (int k = 0; k < 8; ++k) rec.ic[k] = inv_corner(cc.lo, cc.hi, qss, k);
}

// Collimator grid points (kind 2): every other bar counts, one record per thread.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void pair_terms_all_kernel(ScatterLaunch A) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const PeGeom& G = A.geom;
    const int N = G.g.n_det;
    if (tid >= (int64_t)A.n_rows * A.n_pts * A.sub[0] * A.sub[1] * A.sub[2]) return;
    PairIds P;
    pair_ids(A, tid, P);
    PairTerm out{0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    PairRec& rec = A.pair[tid];
    if (below_window_all(A, A.row_cut[P.r], P.qs, P.cc.q)) {  // never read: every voxel's term is below
        rec.t = out;                                          // the window (scatter_kernel tests first)
        return;
    }
    bool near = false;
    SegDir<double> sdw;
    segdir_init<double>(sdw, P.cc.q[0] - P.qs[0], P.cc.q[1] - P.qs[1], P.cc.q[2] - P.qs[2], 0.0, near);
    for (int k = 0; k < N; ++k) {
        if (k == P.d) continue;
        const Bar<double>& bk = G.bars_d[k];
        const double l = leg_chord(bk, sdw, P.qs, P.cc.q);
        out.s_pe += l * bk.mupe;
        out.s_c += l * bk.muc;
    }
    finish_pair(A, P, out, rec);
}

// Inclusive sum over the lanes of a wave (DPP shifts within rows of 16, then the
// rows' last lanes broadcast).
__device__ __forceinline__ int wave_scan(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

// Can the segment from qs along the unit vector u, of length len, meet bar k's
// bounding sphere?  FP32 with margins over its rounding (coordinates to 4e-6,
// squares of distances to 1e-6 of themselves) and over the 0.001 by which the
// chord's small-component branches move the segment; a false answer means the
// reference's chord is 0.
SMG_FN bool leg_may_hit(const float c[3], float diag, const float qs[3], const float u[3], float len) {
    const float x = c[0] - qs[0], y = c[1] - qs[1], z = c[2] - qs[2];
    const float t = x * u[0] + y * u[1] + z * u[2], d2 = x * x + y * y + z * z;
    const float r = 0.5f * diag + 0.01f;
    return d2 - t * t <= r * r + 1e-5f * d2 && t > -r - 1e-5f * tabs(t) && t < len + r + 1e-5f * tabs(t);
}

// Bar-centre, hole-centre and crystal grid points: the bars flagged in the
// bitmap between the scatter point and bar d count (scatter.cu:1343-1401).  A
// wave takes `per` consecutive records (64, or fewer where they are too few to fill
// the chip), one per lane for the window test and the own-bar part.  The bits of the records that any voxel can use are walked by the
// whole wave: a record's words on the smallest power of two of lanes that covers
// them (64 bars: 4 lanes, 16 records a pass; 2,048 bars: 64 lanes, 64 words a
// pass).  The words become a list of bars, those the segment's line passes clear
// of are dropped in FP32, and the others, of all the records together, are traced
// in FP64 64 at a time; each chord above 0 goes to its record's lane, in the order
// of the bits.  Bound by the latency of the words and of the bars' records; a lane
// walking its own record's bits with an FP64 chord for each left most lanes idle
// (bar-centre crystal scatter, 2,048 bars and 32 x 32 voxels: 13.2 ms -> 4.8 ms;
// 64 bars and 16 x 16 voxels: 0.08 ms both; one record a pass there: 0.25 ms).
struct PairWalk {
    double qs[64][3], D[64][3], inv[64][3], len[64];
    uint8_t small[64][4];
    uint32_t pair[128];  // (record << 26) | bar
    uint16_t bar[2048];  // bit within the 64 words
};
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void pair_terms_kernel(ScatterLaunch A, int per) {
    __shared__ PairWalk W;
    const PeGeom& G = A.geom;
    const int N = G.g.n_det;
    const int lane = threadIdx.x;
    const int64_t total = (int64_t)A.n_rows * A.n_pts * A.sub[0] * A.sub[1] * A.sub[2];
    const int64_t tid = (int64_t)blockIdx.x * per + lane;
    const bool valid = lane < per && tid < total;
    PairIds P;
    pair_ids(A, valid ? tid : total - 1, P);
    PairTerm out{0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    // a scatter point inside bar d does not count, and a record below the window
    // for every voxel is never read (scatter_kernel tests first)
    const bool own = A.kind != 1 && P.sbar == P.d;
    const bool use = valid && !own && !below_window_all(A, A.row_cut[P.r], P.qs, P.cc.q);
    const int skip = A.kind == 1 ? P.d : P.sbar;
    int64_t base = 0;
    if (A.kind == 1) {
        base = ((int64_t)P.s * N + P.d) * N;
    } else {
        const int64_t i = P.sbar < P.d ? P.sbar : P.d, j = P.sbar < P.d ? P.d : P.sbar;
        base = (i * N - i * (i + 1) / 2 + j) * N;
    }
    float qf[3], uf[3], lf;
    {
        bool near = false;
        SegDir<double> sd;
        segdir_init<double>(sd, P.cc.q[0] - P.qs[0], P.cc.q[1] - P.qs[1], P.cc.q[2] - P.qs[2], 0.0, near);
        const double l2 = sd.D[0] * sd.D[0] + sd.D[1] * sd.D[1] + sd.D[2] * sd.D[2];
        const double il = l2 > 0.0 ? rsq_fast(l2) : 0.0;
        lf = float(l2 * il);
        for (int k = 0; k < 3; ++k) {
            qf[k] = float(P.qs[k]);
            uf[k] = float(sd.D[k] * il);
            W.qs[lane][k] = P.qs[k];
            W.D[lane][k] = sd.D[k];
            W.inv[lane][k] = sd.inv[k];
            W.small[lane][k] = sd.small[k];
        }
        W.small[lane][3] = (uint8_t)sd.ns;
        W.len[lane] = sd.len;
    }
    __syncthreads();
    int n2 = 0;  // pairs waiting for their FP64 chord
    auto trace = [&](int cnt) {
        // chords of the first cnt (at most 64) waiting pairs
        double l = 0.0, mpe = 0.0, mc = 0.0;
        int e = 0;
        if (lane < cnt) {
            const uint32_t pr = W.pair[lane];
            e = (int)(pr >> 26);
            const Bar<double>& bk = G.bars_d[pr & 0x3ffffffu];
            SegDir<double> sd;
            double qs[3], q[3];
            for (int k = 0; k < 3; ++k) {
                qs[k] = W.qs[e][k];
                sd.D[k] = W.D[e][k];
                sd.inv[k] = W.inv[e][k];
                sd.small[k] = W.small[e][k];
                q[k] = qs[k] + sd.D[k];
            }
            sd.ns = (int8_t)W.small[e][3];
            sd.len = W.len[e];
            sd.tol_d = 0.0;
            l = leg_chord(bk, sd, qs, q);
            mpe = l * bk.mupe;
            mc = l * bk.muc;
        }
        uint64_t m = __ballot(l > 0.0);
        while (m) {  // to the records' lanes, in order
            const int i = __ffsll((unsigned long long)m) - 1;
            m &= m - 1;
            const int o = __builtin_amdgcn_readlane(e, i);
            const double a = readlane_d(mpe, i), c = readlane_d(mc, i);
            if (lane == o) {
                out.s_pe += a;
                out.s_c += c;
            }
        }
    };
    // lanes per record: a power of two that covers its words, so that a small
    // detector's records are taken several at a time
    const int words = (N + 62) >> 5;
    const int sh = words > 32 ? 6 : words > 1 ? 32 - __clz(words - 1) : 0;
    const uint64_t used = __ballot(use);
    const int slot = lane >> sh, sub = lane & ((1 << sh) - 1);
    for (int e0 = 0; e0 < 64; e0 += 64 >> sh) {
        if (((used >> e0) & (~0ull >> (64 - (64 >> sh)))) == 0) continue;  // wave-uniform
        const int me = e0 + slot;
        const int64_t b0 = ((int64_t)__shfl((int)(base >> 32), me) << 32) | (uint32_t)__shfl((int)base, me);
        const int64_t w0 = b0 >> 5, w1 = (b0 + N - 1) >> 5;
        for (int g0 = 0; g0 < words; g0 += 64) {  // at most 64 words
            const int64_t wi = w0 + g0 + sub;
            uint32_t bits = (used >> me & 1) && wi <= w1 ? A.bitmap[wi] : 0u;
            if (wi == w0) bits &= ~0u << (b0 & 31);
            if (wi == w1) bits &= ~0u >> (31 - ((b0 + N - 1) & 31));
            const int cnt = (int)__popc(bits), end = wave_scan(cnt);
            const int n = __builtin_amdgcn_readlane(end, 63);
            for (int at = end - cnt; bits; ++at) {
                W.bar[at] = (uint16_t)(32 * lane + __builtin_ctz(bits));
                bits &= bits - 1;
            }
            const int k0 = (g0 << 5) - (int)(b0 & 31);  // bar of bit 0 of the group's first word
            __syncthreads();
            for (int i0 = 0; i0 < n; i0 += 64) {
                const int v = i0 + lane < n ? W.bar[i0 + lane] : 0;
                const int src = (v >> (5 + sh)) << sh;  // first lane of the entry's group
                const int e = e0 + (v >> (5 + sh));
                const int k = __shfl(k0, src) + (v & ((32 << sh) - 1));
                const float q[3] = {__shfl(qf[0], e), __shfl(qf[1], e), __shfl(qf[2], e)};
                const float u[3] = {__shfl(uf[0], e), __shfl(uf[1], e), __shfl(uf[2], e)};
                const float len = __shfl(lf, e);
                const int d = __shfl(P.d, e), sk = __shfl(skip, e);
                bool hit = false;
                if (i0 + lane < n && k != d && k != sk) {
                    const Bar<float>& bf = G.bars_f[k];
                    const float c[3] = {bf.cx, bf.cy, bf.cz};
                    hit = leg_may_hit(c, bf.rdiag, q, u, len);
                }
                const uint64_t m = __ballot(hit);
                if (hit) W.pair[n2 + (int)__popcll(m & ((1ull << lane) - 1ull))] = ((uint32_t)e << 26) | (uint32_t)k;
                n2 += (int)__popcll(m);
                if (n2 >= 64) {
                    __syncthreads();
                    trace(64);
                    const uint32_t rest = lane < n2 - 64 ? W.pair[64 + lane] : 0u;
                    __syncthreads();
                    n2 -= 64;
                    if (lane < n2) W.pair[lane] = rest;
                }
            }
            __syncthreads();
        }
    }
    __syncthreads();
    trace(n2);
    if (!valid) return;
    PairRec& rec = A.pair[tid];
    if (use)
        finish_pair(A, P, out, rec);
    else
        rec.t = out;
}

// Waves per element row: the scatter points split into `slices` ranges, each
// range summed by its own wave, when rows x voxel waves alone would leave the
// chip under-filled (a few detector rows, or a small image: up to 16,384
// waves), and into up to 16 ranges towards 262,144 waves otherwise.  The
// waves' costs differ widely (the terms that pass the energy window depend on
// the row and the voxels), so short waves shorten the launch's tail: the
// 0.5 mm collimator grid (16,384 unsliced waves per chunk) ran 12% faster
// with 16 slices, its resident waves per SIMD having averaged 1.9 of 3.
struct SliceShape {
    int64_t rows, waves_per_det;
    int slices, per;  // per: scatter points per slice
};

SliceShape slice_shape(const ScatterLaunch& A) {
    SliceShape s;
    s.rows = A.n_rows;
    s.waves_per_det = (A.geom.g.n_vox + 63) / 64;
    const int64_t base = s.rows * s.waves_per_det;
    constexpr int64_t kFillWaves = 16384;     // 256 CUs x 4 SIMDs x 16
    constexpr int64_t kTailWaves = 262144;    // 256 CUs x 4 SIMDs x 256
    constexpr int64_t kTailSlices = 16;
    constexpr int64_t kMinPoints = 32;        // scatter points per wave, at least
    int64_t n = 1;
    if (base > 0)
        n = std::max<int64_t>((kFillWaves + base - 1) / base,
                              std::min<int64_t>(kTailSlices, (kTailWaves + base - 1) / base));
    n = std::min<int64_t>(n, std::max<int64_t>(1, (int64_t)A.n_pts / kMinPoints));
    n = std::max<int64_t>(n, 1);
    s.per = (int)((A.n_pts + n - 1) / n);
    s.slices = s.per > 0 ? (int)((A.n_pts + s.per - 1) / s.per) : 1;
    if (s.slices < 1) s.slices = 1;
    return s;
}

// Per-wave term lists of scatter_kernel, in LDS.  Most terms fail the
// energy-window test, and those that pass are scattered over the lanes, so a
// wave that evaluated the term of every lane for each scatter point in turn
// kept about half its lanes idle.  Instead a batch of scatter points is first
// tested (each lane for its voxel), the (point, lane) pairs that pass are
// listed, the terms of the list are evaluated 64 at a time (lane k takes pair
// k, whatever its voxel), and each lane then adds its own terms in point
// order: the same sums, in the same order, as the per-point loop.
constexpr int kScatterBatchPts = 128;  // points with a passing lane per batch
constexpr int kTestPts = 4;            // points tested per step
template <bool kExact>
struct ScatterLists {
    static constexpr int kCap = kExact ? 512 : 704;  // pairs per batch
    static constexpr int kRedo = kExact ? 1 : 128;   // FP32 terms waiting for FP64
    using T = typename std::conditional<kExact, double, float>::type;
    uint64_t mask[kScatterBatchPts];  // lanes whose term passes, per batch point
    int pre[kScatterBatchPts];        // pairs listed before the point
    int pt[kScatterBatchPts];         // the point's index
    uint16_t pair[kCap];              // (batch point << 6) | lane
    T val[kCap];                      // the pairs' terms
    double vp[3][64];                 // the lanes' voxels
    float4 ptest[64];                 // 64 points: the FP32 window test's vector and limit
    int redo_pt[kRedo];               // the waiting terms' points, and (sub-cell << 6) | lane
    uint32_t redo_at[kRedo];
};

// Ball around the wave's voxels: the middle of their extent and the largest
// distance from it.
__device__ __forceinline__ void wave_ball(const double p[3], bool valid, double C[3], double& R) {
    double d2 = 0.0;
    for (int k = 0; k < 3; ++k) {
        double lo = valid ? p[k] : 1e300, hi = valid ? p[k] : -1e300;
        for (int off = 32; off > 0; off >>= 1) {
            lo = tmin2(lo, __shfl_xor(lo, off));
            hi = tmax2(hi, __shfl_xor(hi, off));
        }
        C[k] = uniform_d(0.5 * (lo + hi));
        d2 += (p[k] - C[k]) * (p[k] - C[k]);
    }
    if (!valid) d2 = 0.0;
    for (int off = 32; off > 0; off >>= 1) d2 = tmax2(d2, __shfl_xor(d2, off));
    R = uniform_d(sqrt(d2) * (1.0 + 1e-9) + 1e-9);
}

// True when the terms of scatter point qs (b = q - qs, nb2 = |b|^2) lie below
// the energy window for every voxel of the ball (C, R): below_window_all for a
// wave's voxels, with cos(alpha - beta), sin(beta) = R / L, from products.
__device__ __forceinline__ bool below_window_ball(double c_lo, const double qs[3], const double b[3], double nb2,
                                                  const double C[3], double R) {
    if (c_lo <= -1.5) return false;  // nothing is rejected
    const double u[3] = {qs[0] - C[0], qs[1] - C[1], qs[2] - C[2]};
    const double L2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    if (!(L2 > R * R * (1.0 + 1e-6) + 1e-9) || !(nb2 > 1e-12)) return false;
    const double iL = rsq_fast(L2);
    const double ca = tmax2(tmin2((u[0] * b[0] + u[1] * b[1] + u[2] * b[2]) * iL * rsq_fast(nb2), 1.0), -1.0);
    const double sb = R * iL, cb = sqrt(tmax2(1.0 - sb * sb, 0.0));
    if (ca >= cb) return false;  // the ball reaches the forward direction
    return ca * cb + sqrt(tmax2(1.0 - ca * ca, 0.0)) * sb < c_lo - 1.1e-4;
}

// kWin: the FP32 term with the row's window table; without one (win_n = 0) it
// evaluates the window probability, and all else is the same (2,048 bars, crystal,
// 511 keV with a 250-650 keV window: 39.2 ms; 64 bars, 1 mm collimator grid over
// 4,096 voxels: 94.2 ms, and with one bar of resolution 0 at 140.5 keV, +-10%, 46.2
// ms against 40.3 with the table).
// Bound by the latency of the terms' FP64 chains and gathers: 168 VGPRs, 3 waves
// per SIMD; a cap of 128 for 4 waves spills as much as the wave gains (1 mm
// collimator grid 237.6 ms against 239.0, crystal grid 20.9 against 19.2).
// Dropping whole points by the wave's ball before the lanes' tests took crystal
// scatter, where 99% of the terms fail, from 28.8 to 25.5 ms; letting FP32 terms
// near a threshold wait for an FP64 loop outside the FP32 one took the grid from
// 262.8 to 246.4 ms (with the inline FP64 term its registers are live across the
// FP32 term).  LDS 9.9 KB per wave.
template <bool kExact, bool kWin>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void scatter_kernel(
    ScatterLaunch A, SliceShape sh) {
    using T = typename std::conditional<kExact, double, float>::type;
    using Lists = ScatterLists<kExact>;
    __shared__ Lists S;
    const PeGeom& G = A.geom;
    const GeomDesc& g = G.g;
    const int lane = threadIdx.x;
    const int64_t waves_per_det = sh.waves_per_det;
    const int64_t wrow = blockIdx.x % (sh.rows * waves_per_det);
    const int slice = (int)(blockIdx.x / (sh.rows * waves_per_det));
    const int r = (int)(wrow / waves_per_det);  // output row
    const int d = row_bar(A, r);
    const int64_t v = (wrow % waves_per_det) * 64 + lane;
    const bool valid = v < g.n_vox;
    const bool sliced = sh.slices > 1;
    float* out = A.dst + (int64_t)r * g.n_vox;
    double* part = A.partial + ((int64_t)slice * sh.rows + r) * g.n_vox;
    const int s_begin = slice * sh.per;
    const int s_end = min(A.n_pts, s_begin + sh.per);
    const Bar<double>& bd = G.bars_d[d];
    if (!A.compton_on || !(bd.mut > (double)0.01f)) {  // scatter.cu:1226-1228
        if (valid) {
            if (sliced)
                part[v] = 0.0;
            else
                out[v] = A.accumulate ? out[v] : 0.0f;
        }
        return;
    }
    const int64_t vv = valid ? v : 0;
    const int nxy = g.nx * g.ny;
    const int iz = (int)(vv / nxy), rem = (int)(vv % nxy);
    double p[3];
    voxel_position(g, rem % g.nx, rem / g.nx, iz, A.cphi, A.sphi, p);

    ScatterPhys ph;
    row_phys(A, bd, ph);
    ph.norm = A.kn_norm;
    ph.inv_norm = uniform_d(1.0 / A.kn_norm);
    ph.tab = A.tables;
    ph.tabf = A.tables_f;
    ph.knp = A.kn_table;
    if constexpr (kWin) {
        const WinRow& w = A.win_rows[r];
        ph.win = A.win_tab + (int64_t)r * A.win_n * 4;
        ph.win_n = A.win_n;
        ph.win_x0 = uniform_d(w.x0);
        ph.win_scale = uniform_d(w.scale);
        ph.omc_lo = uniform_d(w.omc_lo);
        ph.omc_hi = uniform_d(w.omc_hi);
    }
    ph.mupe = bd.mupe;
    ph.muc = bd.muc;
    {
        const double sx = A.sub[0], sy = A.sub[1], sz = A.sub[2];
        ph.rcell = sqrt(bd.w * bd.w / sx / sx + bd.h * bd.h / sz / sz + bd.t * bd.t / sy / sy) / 2.0;
    }
    ph.c_rej = window_cut_margin(A.row_cut[r], kExact ? 1e-9 : 1e-5);  // window_reject_cos(ph, .)
    // the row's physics is the same for every lane: scalar registers
    ph.e0 = uniform_d(ph.e0);
    ph.lo = uniform_d(ph.lo);
    ph.hi = uniform_d(ph.hi);
    ph.norm = uniform_d(ph.norm);
    ph.res = uniform_d(ph.res);
    ph.mupe = uniform_d(ph.mupe);
    ph.muc = uniform_d(ph.muc);
    ph.rcell = uniform_d(ph.rcell);
    ph.c_rej = uniform_d(ph.c_rej);
    const int ncell = A.sub[0] * A.sub[1] * A.sub[2];
    const T wscale = T(bd.muc / bd.mupe);  // crystal weight uses bar d's mu (scatter.cu:1218-1219)
    // scatter points inside bar d itself do not count: its centre (kind 0),
    // or its grid points (kind 3)
    int skip_lo = 0, skip_hi = 0;
    if (A.kind == 0) {
        skip_lo = d;
        skip_hi = d + 1;
    } else if (A.kind == 3) {
        skip_lo = (d - A.pt_bar0) * A.pts_per_bar;
        skip_hi = skip_lo + A.pts_per_bar;
    }
    const int64_t v0 = v - lane;  // first voxel of the wave
    for (int k = 0; k < 3; ++k) S.vp[k][lane] = p[k];
    double C[3], R;
    wave_ball(p, valid, C, R);
    const double c_lo = uniform_d(A.row_cut[r]);
    const float c_rej = float(ph.c_rej);
    // weight of scatter point s for voxel vo at po
    auto weight = [&](int s, int64_t vo, const double po[3]) -> T {
        if (A.kind == 0) return T(A.pe[(int64_t)s * g.n_vox + vo]) * wscale;
        if (A.kind == 2 || A.kind == 3) return T(A.w1[(int64_t)s * g.n_vox + vo]);
        const ScatterPt<double>& sp = A.pts_d[s];
        double dx = po[0] - sp.x, dy = po[1] - sp.y, dz = po[2] - sp.z;
        double lv = sqrt(dx * dx + dy * dy + dz * dz);
        double om;
        if (A.variant == 0) {  // scatter.cu:1711-1716
            double rr = (double)0.1f;
            om = (rr * rr * 3.14159265358979323846 + sp.dy * rr) /
                 (4.0 * 3.14159265358979323846 * lv * lv) * fabs(sp.y - po[1]) / lv;
        } else {  // ScatterGen_Collimator/scatter.cu:1212-1215
            double rr = (double)0.2f;
            om = (rr * rr + sp.dy * rr) / (4.0 * lv * lv);
        }
        return T(om * A.coll_ratio);
    };
    const uint64_t below = (1ull << lane) - 1ull;  // the lanes under this one
    KahanSum<T> acc;
    unsigned fallbacks = 0;
    auto set_cell = [&](int cell, ScatterCell& o) {
        const int a = cell % A.sub[0], b = (cell / A.sub[0]) % A.sub[1], c = cell / (A.sub[0] * A.sub[1]);
        CellCtx cc;
        make_cell_ctx(bd, a, b, c, A.sub[0], A.sub[1], A.sub[2], cc);
        for (int k = 0; k < 3; ++k) {
            o.q[k] = cc.q[k];
            o.lo[k] = cc.lo[k];
            o.hi[k] = cc.hi[k];
        }
    };
    // scatter point si and the voxel of lane o into sk (its sub-cell set
    // before), po and pso; the point's weight for the voxel
    auto set_pair = [&](int si, int o, int cell, ScatterCell& sk, double po[3], double pso[3]) -> T {
        for (int q = 0; q < 3; ++q) po[q] = S.vp[q][o];
        to_frame(bd, po, pso);
        const ScatterPt<double>& sp = A.pts_d[si];
        sk.qs[0] = sp.x;
        sk.qs[1] = sp.y;
        sk.qs[2] = sp.z;
        to_frame(bd, sk.qs, sk.qss);
        const PairRec& rec = A.pair[((int64_t)r * A.n_pts + si) * ncell + cell];
        sk.pt = rec.t;
        sk.ic = rec.ic;
        return weight(si, v0 + o, po);
    };
    ScatterCell sc;          // the current sub-cell
    int cell = -1;
    int s = s_end;           // next point of the range
    int s_blk = s_end;       // first point of the 64 that `live` describes
    uint64_t live = 0;       // of those, the ones still to be tested
    int n = 0, nb = 0;       // the batch: its pairs and its points with a passing lane
    int base = 0;            // its next 64 pairs
    bool more = s_begin < s_end;
    while (more) {  // wave-uniform
        int n_redo = 0;
        while (kExact || n_redo <= Lists::kRedo - 64) {
            if (base >= n) {
                // 3. the finished batch: each lane's terms in point order (a
                // term of weight 0 adds an exact 0)
                __syncthreads();
                for (int j = 0; j < nb; ++j) {
                    const uint64_t m = S.mask[j];
                    if ((m >> lane) & 1ull) acc.add(S.val[S.pre[j] + __popcll(m & below)]);
                }
                __syncthreads();  // the lists are refilled
                n = nb = base = 0;
                if (!live && s >= s_end) {
                    if (++cell >= ncell) {
                        more = false;
                        break;
                    }
                    s = s_begin;
                    set_cell(cell, sc);
                    for (int k = 0; k < 3; ++k) {  // the same for every lane
                        sc.q[k] = uniform_d(sc.q[k]);
                        sc.lo[k] = uniform_d(sc.lo[k]);
                        sc.hi[k] = uniform_d(sc.hi[k]);
                    }
                }
                // 1. the next batch: points in order until kScatterBatchPts of
                // them have a passing lane or the list could overflow with the
                // next ones.  Points go through 64 at a time, lane l looking at
                // point s_blk + l: those below the window for every voxel of the
                // wave are dropped, and the others leave b = q - qs and the
                // limit of the lanes' test.
                while (nb <= kScatterBatchPts - kTestPts && n <= Lists::kCap - 64 * kTestPts) {
                    if (!live) {
                        if (s >= s_end) break;
                        s_blk = s;
                        s = min(s + 64, s_end);
                        const int si = s_blk + lane;
                        bool keep = si < s && !(si >= skip_lo && si < skip_hi);
                        if (keep) {
                            const ScatterPt<double>& sp = A.pts_d[si];
                            const double qs[3] = {sp.x, sp.y, sp.z};
                            const double bq[3] = {sc.q[0] - qs[0], sc.q[1] - qs[1], sc.q[2] - qs[2]};
                            const double nb2 = bq[0] * bq[0] + bq[1] * bq[1] + bq[2] * bq[2];
                            keep = !below_window_ball(c_lo, qs, bq, nb2, C, R);
                            // a.b < c |a| |b| as signed squares: a.b |a.b| < (c |c| |b|^2) |a|^2
                            S.ptest[lane] = make_float4(float(bq[0]), float(bq[1]), float(bq[2]),
                                                        c_rej * tabs(c_rej) * float(nb2));
                        }
                        live = __ballot(keep);
                        __syncthreads();
                        continue;
                    }
                    // kTestPts points at a time, their data fetched together
                    int pi[kTestPts];
                    double qx[kTestPts], qy[kTestPts], qz[kTestPts];
                    float4 t[kTestPts];
                    bool on[kTestPts];
#pragma unroll
                    for (int u = 0; u < kTestPts; ++u) {
                        on[u] = live != 0;
                        pi[u] = on[u] ? __ffsll((unsigned long long)live) - 1 : (u ? pi[u - 1] : 0);
                        if (on[u]) live &= live - 1;
                        const ScatterPt<double>& sp = A.pts_d[s_blk + pi[u]];
                        qx[u] = sp.x;
                        qy[u] = sp.y;
                        qz[u] = sp.z;
                        if constexpr (!kExact) t[u] = S.ptest[pi[u]];
                    }
#pragma unroll
                    for (int u = 0; u < kTestPts; ++u) {
                        bool pass;
                        if constexpr (kExact) {
                            sc.qs[0] = qx[u];
                            sc.qs[1] = qy[u];
                            sc.qs[2] = qz[u];
                            pass = valid && on[u] && !below_window<T>(ph, p, sc);
                        } else {
                            const float ax = float(qx[u] - p[0]), ay = float(qy[u] - p[1]), az = float(qz[u] - p[2]);
                            const float ab = ax * t[u].x + ay * t[u].y + az * t[u].z;
                            pass = valid && on[u] && !(ab * tabs(ab) < t[u].w * (ax * ax + ay * ay + az * az));
                        }
                        const uint64_t m = __ballot(pass);
                        if (m) {  // wave-uniform
                            if (pass) S.pair[n + __popcll(m & below)] = (uint16_t)((nb << 6) | lane);
                            if (lane == 0) {
                                S.mask[nb] = m;
                                S.pre[nb] = n;
                                S.pt[nb] = s_blk + pi[u];
                            }
                            n += __popcll(m);
                            ++nb;
                        }
                    }
                }
                __syncthreads();
                continue;
            }
            // 2. the batch's next 64 terms
            const int k = base + lane;
            base += 64;
            bool near = false;
            int at = 0, si = 0;
            if (k < n) {
                const int e = S.pair[k];
                at = e & 63;
                si = S.pt[e >> 6];
                ScatterCell sk;
                double po[3], pso[3];
                for (int q = 0; q < 3; ++q) {
                    sk.q[q] = sc.q[q];
                    sk.lo[q] = sc.lo[q];
                    sk.hi[q] = sc.hi[q];
                }
                const T wgt = set_pair(si, at, cell, sk, po, pso);
                T val = T(0);
                if (wgt != T(0)) val = scatter_term<T, true, kWin>(ph, po, pso, sk, wgt, near);
                S.val[k] = (!kExact && near) ? T(0) : val;
            }
            if constexpr (!kExact) {
                // an FP32 term near a threshold waits for FP64
                const uint64_t m = __ballot(near);
                if (m) {  // wave-uniform
                    if (near) {
                        const int i = n_redo + __popcll(m & below);
                        S.redo_pt[i] = si;
                        S.redo_at[i] = ((uint32_t)cell << 6) | (uint32_t)at;
                    }
                    n_redo += __popcll(m);
                }
            }
        }
        if constexpr (!kExact) {
            // the waiting terms, outside the loop above so that their FP64
            // registers are not live in it; each goes to its voxel's lane, in
            // list order
            __syncthreads();
            for (int i0 = 0; i0 < n_redo; i0 += 64) {
                const int i = i0 + lane;
                double val = 0.0;
                int at = 0;
                if (i < n_redo) {
                    const int c = (int)(S.redo_at[i] >> 6);
                    at = (int)(S.redo_at[i] & 63u);
                    ScatterCell sk;
                    double po[3], pso[3];
                    set_cell(c, sk);
                    const T wgt = set_pair(S.redo_pt[i], at, c, sk, po, pso);
                    bool n2 = false;
                    val = scatter_term<double, true>(ph, po, pso, sk, double(wgt), n2);
                    ++fallbacks;
                }
                const int cnt = min(64, n_redo - i0);
                for (int e = 0; e < cnt; ++e) {
                    const double x = __shfl(val, e);
                    if (lane == __shfl(at, e)) acc.add(T(x));
                }
            }
            __syncthreads();
        }
    }
    if (valid) {
        if (sliced)
            part[v] = double(acc.s) + double(acc.c);
        else
            out[v] = A.accumulate ? out[v] + float(acc.value()) : float(acc.value());
    }
    if constexpr (!kExact) {
        unsigned tot = fallbacks;
        for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
        if (lane == 0 && tot) atomicAdd(&A.counters[0], (unsigned long long)tot);
    }
}

// The KN prefix polynomials of alpha, one block: thread k forms node k of every
// phase, one thread per phase sums them in order, thread k expands its
// polynomial.
__global__ __launch_bounds__(kKnSteps) void kn_table_kernel(double alpha, double* tab) {
    __shared__ double node[kKnDeg + 1][kKnSteps];
    const int k = threadIdx.x;
    for (int m = 0; m <= kKnDeg; ++m) node[m][k] = kn_node(alpha, kn_phase(m), k);
    __syncthreads();
    if (k <= kKnDeg) {
        KahanSum<double> s;
        for (int i = 0; i < kKnSteps; ++i) {
            s.add(node[k][i]);
            node[k][i] = s.value();
        }
    }
    __syncthreads();
    double v[kKnDeg + 1], c[kKnDeg + 1];
    for (int m = 0; m <= kKnDeg; ++m) v[m] = node[m][k];
    kn_poly_coeffs(v, c);
    for (int j = 0; j < kKnStride; ++j) tab[(size_t)k * kKnStride + j] = j <= kKnDeg ? c[j] : 0.0;
}

// Sum of the slices' partial sums of one element, in slice order (a fixed
// order, so the result does not depend on scheduling), compensated in FP64.
__global__ __launch_bounds__(256) void scatter_reduce_kernel(ScatterLaunch A, SliceShape sh) {
    const int64_t n_vox = A.geom.g.n_vox;
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = sh.rows * n_vox;
    if (tid >= n) return;
    KahanSum<double> acc;
    for (int k = 0; k < sh.slices; ++k) acc.add(A.partial[(int64_t)k * n + tid]);
    const float val = float(acc.value());
    A.dst[tid] = A.accumulate ? A.dst[tid] + val : val;
}

// Grid scatterers (an extension with no reference counterpart): one thread
// per (scatter point s, voxel v) of the chunk, the chance of a Compton
// interaction in the cell around s for a photon from v,
// w_s / (4 pi |s - v|^2) exp(-collimator material along v -> s), in FP64,
// with w_s = dv mu_c of the point's layer (held in the point's dy).
__global__ __launch_bounds__(256) void first_leg_kernel(ScatterLaunch A, float* w1) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const GeomDesc& g = A.geom.g;
    const int64_t total = (int64_t)A.n_pts * g.n_vox;
    if (tid >= total) return;
    const int s = (int)(tid / g.n_vox);
    const int64_t v = tid % g.n_vox;
    const int nxy = g.nx * g.ny;
    const int iz = (int)(v / nxy), rem = (int)(v % nxy);
    double p[3];
    voxel_position(g, rem % g.nx, rem / g.nx, iz, A.cphi, A.sphi, p);
    const ScatterPt<double>& sp = A.pts_d[s];
    const double q[3] = {sp.x, sp.y, sp.z};
    double att_t, s_pe, s_c;
    coll_material(A.geom, p, q, att_t, s_pe, s_c);
    const double dx = q[0] - p[0], dy = q[1] - p[1], dz = q[2] - p[2];
    const double L2 = dx * dx + dy * dy + dz * dz;
    w1[tid] = float(sp.dy / (4.0 * 3.14159265358979323846 * L2) * exp(-att_t));
}

}  // namespace

hipError_t launch_first_leg(const ScatterLaunch& A, float* w1, hipStream_t stream) {
    const int64_t total = (int64_t)A.n_pts * A.geom.g.n_vox;
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(first_leg_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream,
                       A, w1);
    return hipGetLastError();
}

hipError_t launch_kn_table(double e0, double* tab, hipStream_t stream) {
    hipLaunchKernelGGL(kn_table_kernel, dim3(1), dim3(kKnSteps), 0, stream, e0 / 511.0, tab);
    return hipGetLastError();
}

hipError_t launch_row_cuts(const ScatterLaunch& A, double* cut, WinRow* win, float* tab, hipStream_t stream) {
    const int64_t rows = A.n_rows;
    if (rows <= 0) return hipSuccess;
    if (A.win_n > 0 && (!win || !tab)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(row_cut_kernel, dim3((unsigned)((rows + 63) / 64)), dim3(64), 0, stream, A, cut, win);
    if (A.win_n > 0)
        hipLaunchKernelGGL(win_table_kernel, dim3((unsigned)((rows * A.win_n + 255) / 256)), dim3(256), 0, stream, A,
                           win, tab);
    return hipGetLastError();
}

hipError_t launch_pair_terms(const ScatterLaunch& A, hipStream_t stream) {
    const int64_t rows = A.n_rows;
    const int64_t total = rows * A.n_pts * A.sub[0] * A.sub[1] * A.sub[2];
    if (total <= 0) return hipSuccess;
    if (A.kind == 2) {
        hipLaunchKernelGGL(pair_terms_all_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, A);
        return hipGetLastError();
    }
    // 2,048 waves (2 per SIMD) where the records allow it, of 8 records at least: a
    // wave's passes over its records are one chain of latencies (160 bars, one hole, 3
    // sub-cells, 480 records: 170 us at 64 a wave, call 300 us; 160 us at 8; 256 bars
    // crystal, 65,536 records: 50 us at 64, 40 at 32)
    int per = 64;
    while (per > 8 && total <= (int64_t)(per / 2) * 2048) per /= 2;
    hipLaunchKernelGGL(pair_terms_kernel, dim3((unsigned)((total + per - 1) / per)), dim3(64), 0, stream, A, per);
    return hipGetLastError();
}

size_t scatter_partial_size(const ScatterLaunch& A) {
    const SliceShape sh = slice_shape(A);
    return sh.slices > 1 ? (size_t)sh.slices * (size_t)sh.rows * (size_t)A.geom.g.n_vox : 0;
}

hipError_t launch_scatter(const ScatterLaunch& A, bool exact, hipStream_t stream) {
    const SliceShape sh = slice_shape(A);
    const int64_t blocks = sh.slices * sh.rows * sh.waves_per_det;
    if (blocks <= 0) return hipSuccess;
    if (sh.slices > 1 && !A.partial) return hipErrorInvalidValue;
    if (exact)
        hipLaunchKernelGGL((scatter_kernel<true, false>), dim3((unsigned)blocks), dim3(64), 0, stream, A, sh);
    else if (A.win_n > 0)
        hipLaunchKernelGGL((scatter_kernel<false, true>), dim3((unsigned)blocks), dim3(64), 0, stream, A, sh);
    else
        hipLaunchKernelGGL((scatter_kernel<false, false>), dim3((unsigned)blocks), dim3(64), 0, stream, A, sh);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || sh.slices == 1) return e;
    const int64_t n = sh.rows * A.geom.g.n_vox;
    hipLaunchKernelGGL(scatter_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       A, sh);
    return hipGetLastError();
}

namespace {

// out = a + b, four floats per thread where the three pointers allow it.
__global__ __launch_bounds__(256) void add_blocks_kernel(const float* a, const float* b, float* out,
                                                         size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = a[i] + b[i];
}

__global__ __launch_bounds__(256) void add_blocks4_kernel(const float4* a, const float4* b, float4* out,
                                                          size_t n4) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
        const float4 x = a[i], y = b[i];
        out[i] = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
    }
}

}  // namespace

hipError_t launch_add_blocks(const float* a, const float* b, float* out, size_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const bool al = ((uintptr_t)a | (uintptr_t)b | (uintptr_t)out) % 16 == 0 && n % 4 == 0;
    const size_t work = al ? n / 4 : n;
    const unsigned blocks = (unsigned)std::min<size_t>((work + 255) / 256, 8192);
    if (al)
        hipLaunchKernelGGL(add_blocks4_kernel, dim3(blocks), dim3(256), 0, stream, (const float4*)a,
                           (const float4*)b, (float4*)out, work);
    else
        hipLaunchKernelGGL(add_blocks_kernel, dim3(blocks), dim3(256), 0, stream, a, b, out, n);
    return hipGetLastError();
}

}  // namespace smg
