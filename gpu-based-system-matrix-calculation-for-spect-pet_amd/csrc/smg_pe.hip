// Photoelectric system-matrix kernel for gfx950 (CDNA4, wave64).
//
// Work decomposition: one wave per (detector bar d, tile of 64 voxels).  The
// reference runs one thread per (d, v) and makes every thread scan all bars
// and holes for culling (PEGen_RayTracing_CircularHole/PESysMatGen.cu:1097-1186)
// before its sub-cell loop (:1193-1362).  Here the 64 lanes of a wave share
// detector d, so every sub-cell point is wave-uniform and:
//   1. the wave scans the bars and holes once, 64 at a time, keeping those
//      whose box a segment from bar d to the tile can meet (any other has
//      chord 0 for every ray of the wave, so whether the reference would cull
//      it does not change the result), with the lanes whose reference culling
//      predicate keeps them, in LDS;
//   2. for a block of sub-cells at once, the candidates are narrowed to those
//      whose box can meet a segment from the sub-cell centre to the tile (a bar
//      outside that cone has chord 0 for every lane, so dropping it is exact),
//      and the records of the kept (sub-cell, candidate) pairs are formed in LDS;
//   3. every lane traces its own ray against the narrowed lists (wave-uniform
//      loops, per-lane masks) and accumulates the sub-cell terms with a
//      two-sum compensated sum;
//   4. each lane writes its element once: no atomics, deterministic results.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "smg_kernels.hpp"
#include "smg_pe_body.hpp"

namespace smg {

namespace {

// Sub-cells of one block of the narrowing, at most (one lane holds each).
constexpr int kBlockCells = 64;
// Room for (sub-cell, candidate) records beside full candidate lists, in
// 8-byte words.
constexpr int kRecWords = 244;

// Candidate lists of one wave, in LDS, for up to CapB bars and CapH holes.
// arena: the lane masks of the n = nb + nh candidates of the tile (bars first,
// then holes), then the records of the narrowed pairs: bars upward from word n,
// holes downward from the end.  The lists are short as a rule (about 27
// candidates on the full-size geometry), so the records of a whole block fit.
template <int CapB, int CapH, bool kShared = false>
struct WaveListsT {
    static constexpr int cap_bars = CapB, cap_holes = CapH;
    static constexpr int arena_words = CapB + CapH + kRecWords;
    static constexpr int sel_cap = 64;
    uint64_t arena[CapB + CapH + kRecWords];
    uint64_t sel[sel_cap];       // per sub-cell of the block: the candidates it keeps
    uint64_t redo[kBlockCells];  // per sub-cell of the block: the lanes to redo in FP64
    uint16_t idx[CapB + CapH];   // bar or hole number of each candidate
    // kShared: the block has several waves, each with lists of its own.  A wave's
    // LDS accesses are in order: only the compiler has to keep them so.
    __device__ static void sync() {
        if constexpr (kShared) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    }
};
using WaveLists = WaveListsT<kCapBars, kCapHoles>;
using SharedLists = WaveListsT<kCapBars, kCapHoles, true>;

// The adjoint's lists hold fewer bars: with its per-candidate FP64 sums and
// kept chords, 13 KB of LDS per wave, so 12 waves (3 per SIMD) fit a CU.
constexpr int kCapBarsAdjoint = 320;
using AdjointLists = WaveListsT<kCapBarsAdjoint, kCapHoles>;

// Candidate lists of a wave whose tile overflowed the LDS lists, in its own
// slot of global memory with room for every bar and hole of the geometry (so
// they cannot overflow), plus the adjoint's per-candidate sums.
struct SpillLists {
    int cap_bars, cap_holes, arena_words, sel_cap;
    uint64_t* arena;
    uint64_t* sel;
    uint64_t* redo;
    double* cand_acc;
    uint16_t* idx;
    __device__ static void sync() { __syncthreads(); }
};

__device__ __forceinline__ SpillLists spill_lists(const PeSpill& S, int slot) {
    unsigned char* p = S.slots + (int64_t)slot * S.slot_bytes;
    const int n = S.cap_bars + S.cap_holes;
    SpillLists L;
    L.cap_bars = S.cap_bars;
    L.cap_holes = S.cap_holes;
    L.arena_words = pe_spill_arena_words(S.cap_bars, S.cap_holes);
    L.sel_cap = pe_spill_sel_words(S.cap_bars, S.cap_holes);
    L.arena = (uint64_t*)p;
    p += sizeof(uint64_t) * L.arena_words;
    L.sel = (uint64_t*)p;
    p += sizeof(uint64_t) * L.sel_cap;
    L.redo = (uint64_t*)p;
    p += sizeof(uint64_t) * kBlockCells;
    L.cand_acc = (double*)p;
    p += sizeof(double) * S.cap_bars;
    L.idx = (uint16_t*)p;
    return L;
}

// A wave whose candidates overflowed its LDS lists queues its work item for
// the spill kernel of the same launch; without a queue (a launch with no
// spill area) it is only counted.
__device__ __forceinline__ void spill_push(const PeLaunch& A, int item, int lane) {
    if (lane == 0) {
        const unsigned long long i = atomicAdd(&A.counters[2], 1ull);
        if (A.spill.queue) A.spill.queue[i] = item;
    }
}

// A 64-bit value every lane holds alike, in scalar registers; and its bit of
// this lane, which is the wave's execution mask itself.
__device__ __forceinline__ uint64_t uniform_u64(uint64_t x) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)x);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ bool lane_bit(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// Set bits of m, as a signed number: the hole records are indexed downward
// (__popcll is unsigned, and a negated unsigned index wraps at 2^32).
__device__ __forceinline__ int bit_count(uint64_t m) { return (int)__popcll(m); }

// One sub-cell's narrowed candidates for the lanes of a wave, from its records
// (the FP32 rays).
template <class Lists>
struct RecCands {
    static constexpr bool kFastFaces = true;
    static constexpr bool kHoleRecs = true;
    const Lists* L;
    const BarRec* b;   // record j: b[j]
    const HoleRec* h;  // record j: h[-j]
    int nb, nh;
    __device__ int nbars() const { return nb; }
    __device__ bool fast(int j) const { return b[j].tag & kFastBar; }
    __device__ const float* faces(int j) const { return b[j].face; }
    __device__ double mu(int j) const { return b[j].mu; }
    __device__ int pos(int j) const { return b[j].tag & 0xffff; }
    // the index is wave-uniform: readfirstlane lets the record loads go
    // through the scalar unit
    __device__ int bar(int j) const { return __builtin_amdgcn_readfirstlane(L->idx[pos(j)]); }
    __device__ bool bar_on(int j) const { return lane_bit(uniform_u64(b[j].lanes)); }
    __device__ int nholes() const { return nh; }
    __device__ const HoleRec& hole_rec(int j) const { return h[-j]; }
    __device__ int hole(int j) const { return __builtin_amdgcn_readfirstlane(h[-j].hole); }
    __device__ bool hole_on(int j) const { return lane_bit(uniform_u64(h[-j].lanes)); }
};

// The same from the positions of the candidates in the list (the FP64 rays).
template <class Lists>
struct ListCands {
    static constexpr bool kFastFaces = false;
    const Lists* L;
    const uint16_t* cur;  // bars, then holes
    int nb, nh;
    __device__ int nbars() const { return nb; }
    __device__ int pos(int j) const { return cur[j]; }
    __device__ int bar(int j) const { return __builtin_amdgcn_readfirstlane(L->idx[cur[j]]); }
    __device__ bool bar_on(int j) const { return lane_bit(uniform_u64(L->arena[cur[j]])); }
    __device__ int nholes() const { return nh; }
    __device__ int hole(int j) const { return __builtin_amdgcn_readfirstlane(L->idx[cur[nb + j]]); }
    __device__ bool hole_on(int j) const { return lane_bit(uniform_u64(L->arena[cur[nb + j]])); }
};

// Lane and tile state of one wave: voxel of the lane, tile bounding sphere
// and the self-culling terms of bar d.
struct WaveSetup {
    int ix, iy, iz;
    bool valid;
    int64_t v;
    double p[3], ps[3];
    float pf[3];
    SelfCull sc;
    float udf[3], critf;
    double tc[3], rho;
    float tcf[3], te[3];  // tile centre and half extents along the world axes
    uint32_t bar_gate;  // bit m: no ray from bar d to the tile can be stopped by layer m's gate
};

__device__ __forceinline__ void wave_setup(const PeLaunch& A, int d, int tile, int lane, WaveSetup& W) {
    const PeGeom& G = A.geom;
    const GeomDesc& g = G.g;
    const Bar<double>& bd = G.bars_d[d];
    const int t0 = tile % A.tiles[0];
    const int t1 = (tile / A.tiles[0]) % A.tiles[1];
    const int t2 = tile / (A.tiles[0] * A.tiles[1]);
    const int ix0 = t0 * A.tile[0], iy0 = t1 * A.tile[1], iz0 = t2 * A.tile[2];
    W.ix = ix0 + lane % A.tile[0];
    W.iy = iy0 + (lane / A.tile[0]) % A.tile[1];
    W.iz = iz0 + lane / (A.tile[0] * A.tile[1]);
    W.valid = W.ix < g.nx && W.iy < g.ny && W.iz < g.nz;
    W.v = (int64_t)W.ix + (int64_t)W.iy * g.nx + (int64_t)W.iz * g.nx * g.ny;
    voxel_position(g, W.valid ? W.ix : ix0, W.valid ? W.iy : iy0, W.valid ? W.iz : iz0, A.cphi,
                   A.sphi, W.p);
    to_frame(bd, W.p, W.ps);
    for (int k = 0; k < 3; ++k) W.pf[k] = float(W.p[k]);
    self_cull(bd, W.p, W.sc);
    for (int k = 0; k < 3; ++k) W.udf[k] = float(W.sc.ud[k]);
    W.critf = float(W.sc.crit);
    tile_ball(g, ix0, iy0, iz0, A.tile, A.cphi, A.sphi, W.tc, W.rho);
    for (int k = 0; k < 3; ++k) W.tc[k] = uniform_d(W.tc[k]);
    W.rho = uniform_d(W.rho);
    tile_extents(g, ix0, iy0, iz0, A.tile, A.cphi, A.sphi, W.te);
    for (int k = 0; k < 3; ++k) {
        W.tcf[k] = uniform_f(float(W.tc[k]));
        W.te[k] = uniform_f(W.te[k]);
    }
    // plate gates that no ray from any point of bar d (inside its bounding
    // ball, the half diagonal with a rounding margin) to the tile can trigger
    const double qc[3] = {bd.cx, bd.cy, bd.cz};
    const double rb = 0.5 * bd.rdiag * (1.0 + 1e-12) + 1e-9;
    const bool clear = lane < g.n_layers &&
                       plate_gate_clear_ball(G.layers_d[lane < g.n_layers ? lane : 0], qc, rb, W.tc, W.rho);
    W.bar_gate = (uint32_t)__ballot(clear);
    if (bd.sb == 0.0 && bd.cb == 1.0) W.bar_gate |= kUnturned;
    W.bar_gate = __builtin_amdgcn_readfirstlane(W.bar_gate);
}

// Appends the passing lanes' candidates (numbers base + lane) to the list at
// position n.  all: the culling test keeps the candidate for every lane (then
// its mask is the valid lanes'); the others are tested per lane, one after the
// other, and dropped when no lane keeps them.  keep(k): this lane's culling test of
// candidate k.  All are stored at once, each by its lane: a group with one open
// candidate stored one by one took a 2,048-bar panel turned by 0.2 rad, one sub-cell,
// 1 mm voxels 1.73 ms instead of 1.65, a 40x36x12-voxel projection and back
// projection 36.3 instead of 34.6 with the frustum_cut of two selects.
template <class Lists, class Keep>
__device__ __forceinline__ void append_candidates(Lists& L, int cap, int first, int base, bool pass, bool all,
                                                  uint64_t valid, int lane, int& n, Keep keep) {
    uint64_t mask = 0;
    for (uint64_t open = __ballot(pass && !all); open; open &= open - 1) {
        const int bit = __ffsll((unsigned long long)open) - 1;
        const uint64_t m = __ballot(keep(base + bit));
        if (lane == bit) mask = m, pass = m != 0;
    }
    const uint64_t bal = __ballot(pass);
    const int pos = n + bit_count(bal & ((1ull << lane) - 1ull));
    if (pass && pos < cap) {
        L.idx[first + pos] = (uint16_t)(base + lane);
        L.arena[first + pos] = all ? valid : mask;
    }
    n += bit_count(bal);
}

// Step 1: candidate bars and holes of the tile: those whose box a segment from
// bar d to the tile can meet (bar_tile_may_hit with the tile's half extents per
// axis, which are what bounds the scan: a ball around a 4x4x4 tile is 1.7 times
// as wide, and around an 8x8x1 tile 1.4 times along x and y and 2.5 mm instead
// of 0 along z; with the ball the full-size PE step took 187.5 ms instead of
// 177.4, one slice at 8x16x8 sub-cells 37.4 instead of 33.5; first on the box of each
// group of kGroup consecutive bars or holes, then on the members of the
// groups it keeps; any other has chord 0 for every ray of the tile, so its
// culling decision does not matter), each with the lanes whose reference
// culling test keeps it: all of them where cull_keeps_all shows so for the
// tile (99.97% of the candidates on the full-size geometry), else by a ballot
// of the lanes' tests.  kFew (the kernels for few sub-cells, where this scan is
// most of the work, and the adjoint, 64 bars 288 -> 286 us): no cull_keeps_all in
// groups whose members all fail, of which a panel turned by 0.25 rad scans several a
// tile (2.59 -> 2.45 ms at one sub-cell); in the other kernels the branch costs 2%
// (full-size step 128.3 -> 130.5 ms).
// Returns false on overflow.
template <bool kExact, bool kFew, class Lists>
__device__ bool build_candidates(const PeLaunch& A, int d, int lane, const WaveSetup& W,
                                 Lists& L, int& nb, int& nh) {
    const PeGeom& G = A.geom;
    const GeomDesc& g = G.g;
    const Bar<float>& bdf = G.bars_f[d];
    const float cd[3] = {bdf.cx, bdf.cy, bdf.cz};
    const float rho = float(W.rho) * 1.0001f;
    const uint64_t valid = __ballot(W.valid);
    nb = 0;
    nh = 0;
    // groups of kGroup bars first (one group box per lane), then the members
    // of each group that can be hit
    const int n_bg = (g.n_det + kGroup - 1) / kGroup;
    for (int g0 = 0; g0 < n_bg; g0 += 64) {
        bool gpass = false;
        if (g0 + lane < n_bg) {
            const GroupBox& B = G.bar_groups[g0 + lane];
            gpass = bar_tile_may_hit(bdf, W.tcf, W.te, B.c[0], B.c[1], B.c[2], 1.0f, 0.0f, B.h[0],
                                     B.h[1], B.h[2]);
        }
        uint64_t gbal = __ballot(gpass);
        while (gbal) {
            const int base = (g0 + __ffsll((unsigned long long)gbal) - 1) * kGroup;
            gbal &= gbal - 1;
            const int k = base + lane;
            bool pass = false, all = false;
            if (k < g.n_det && k != d) {
                const Bar<float>& b = G.bars_f[k];
                float rt[3];
                extents_in_frame(W.te, b.cb, b.sb, rt);
                pass = bar_tile_may_hit(bdf, W.tcf, rt, b.cx, b.cy, b.cz, b.cb, b.sb, 0.5f * b.w,
                                        0.5f * b.t, 0.5f * b.h);
                const float c[3] = {b.cx, b.cy, b.cz};
                all = (!kFew || pass) && cull_keeps_all(W.tcf, rho, c, 0.5f * b.rdiag, cd, 0.5f * bdf.rdiag);
            }
            append_candidates(L, L.cap_bars, 0, base, pass, all, valid, lane, nb, [&](int kk) {
                return W.valid && cull_bar<kExact>(G, kk, W.p, W.pf, W.sc, W.udf, W.critf);
            });
        }
    }
    if (nb > L.cap_bars) return false;
    const int n_hg = (g.n_holes + kGroup - 1) / kGroup;
    for (int g0 = 0; g0 < n_hg; g0 += 64) {
        bool gpass = false;
        if (g0 + lane < n_hg) {
            const GroupBox& B = G.hole_groups[g0 + lane];
            gpass = bar_tile_may_hit(bdf, W.tcf, W.te, B.c[0], B.c[1], B.c[2], 1.0f, 0.0f, B.h[0],
                                     B.h[1], B.h[2]);
        }
        uint64_t gbal = __ballot(gpass);
        while (gbal) {
            const int base = (g0 + __ffsll((unsigned long long)gbal) - 1) * kGroup;
            gbal &= gbal - 1;
            const int h = base + lane;
            bool pass = false, all = false;
            if (h < g.n_holes) {
                const Hole<float>& o = G.holes_f[h];
                pass = bar_tile_may_hit(bdf, W.tcf, W.te, o.xc, o.ymid, o.zc, 1.0f, 0.0f, o.r,
                                        0.5f * tabs(o.y2 - o.y1), o.r);
                const float c[3] = {o.xc, o.ymid, o.zc};
                all = (!kFew || pass) && cull_keeps_all(W.tcf, rho, c, o.crit, cd, 0.5f * bdf.rdiag);
            }
            append_candidates(L, L.cap_holes, nb, base, pass, all, valid, lane, nh, [&](int hh) {
                return W.valid && cull_hole<kExact>(G, hh, W.p, W.pf, W.sc, W.udf, W.critf);
            });
        }
    }
    return nh <= L.cap_holes;
}

// Sub-cell `cell` of bar d for this wave's tile (from the sub-cell table when
// there is one: wave-uniform, so through the scalar unit), with the plate gates
// that no ray of the tile can trigger: those cleared for the whole bar, else
// tested for the sub-cell point (one layer per lane, then a ballot).
__device__ __forceinline__ void tile_cell(const PeLaunch& A, const Bar<double>& bd, int d, int cell,
                                          const WaveSetup& W, int lane, CellCtx& cc) {
    if (A.cells) {
        typedef const __attribute__((address_space(4))) CellCtx ScalarCell;
        const int64_t i = (int64_t)(d - A.cells_bar0) * (A.sub[0] * A.sub[1] * A.sub[2]) + cell;
        ScalarCell* c = (ScalarCell*)(A.cells + i);
        for (int k = 0; k < 3; ++k) {
            cc.q[k] = c->q[k];
            cc.qs[k] = c->qs[k];
            cc.lo[k] = c->lo[k];
            cc.hi[k] = c->hi[k];
            cc.area[k] = c->area[k];
            cc.hc[k] = c->hc[k];
        }
    } else {
        make_cell_ctx_linear(bd, cell, A.sub, cc);
        for (int k = 0; k < 3; ++k) {
            cc.q[k] = uniform_d(cc.q[k]);
            cc.qs[k] = uniform_d(cc.qs[k]);
            cc.lo[k] = uniform_d(cc.lo[k]);
            cc.hi[k] = uniform_d(cc.hi[k]);
            cc.area[k] = uniform_d(cc.area[k]);
            cc.hc[k] = uniform_f(cc.hc[k]);
        }
    }
    const GeomDesc& g = A.geom.g;
    const uint32_t all = (uint32_t)((1ull << g.n_layers) - 1ull);
    if ((W.bar_gate & all) == all) {  // wave-uniform
        cc.gate_clear = W.bar_gate;  // with its kUnturned bit
        return;
    }
    const bool clear = lane < g.n_layers && !((W.bar_gate >> lane) & 1u) &&
                       plate_gate_clear(A.geom.layers_d[lane < g.n_layers ? lane : 0], cc.q, W.tc, W.rho);
    cc.gate_clear = W.bar_gate | (uint32_t)__ballot(clear);
}

// Centre of this lane's sub-cell `cell` of bar d.
__device__ __forceinline__ void cell_point(const PeLaunch& A, const Bar<double>& bd, int d, int cell, double q[3]) {
    if (A.cells) {
        const CellCtx& c = A.cells[(int64_t)(d - A.cells_bar0) * (A.sub[0] * A.sub[1] * A.sub[2]) + cell];
        for (int k = 0; k < 3; ++k) q[k] = c.q[k];
    } else {
        CellCtx c;
        make_cell_ctx_linear(bd, cell, A.sub, c);
        for (int k = 0; k < 3; ++k) q[k] = c.q[k];
    }
}

// Step 2: the candidates whose box a segment from a sub-cell centre to the
// tile can meet (box_meets_frustum with a point source), for ns sub-cells at
// once (lane s holds the number of the s-th in my_cell): bit j % 64 of
// sel[s * words + j / 64] for candidate j.  A lane keeps one candidate's box for
// all of them, and with at most 32 candidates a pass takes several sub-cells.
// (One sub-cell per pass, its candidates' records gathered anew for each, was a
// quarter of the PE kernel's instructions and most of its waits: full-size step
// 177.4 ms, with this form 169.8; 64-bar slice, one wave per SIMD, 274 -> 246 us.)
template <class Lists>
__device__ __forceinline__ void select_cells(const PeLaunch& A, const Bar<double>& bd, int d, int my_cell, int ns,
                                             const WaveSetup& W, int lane, Lists& L, int nb, int n, int words) {
    const PeGeom& G = A.geom;
    float q0 = 0.0f, q1 = 0.0f, q2 = 0.0f;
    if (lane < ns) {
        double q[3];
        cell_point(A, bd, d, my_cell, q);
        q0 = float(q[0]);
        q1 = float(q[1]);
        q2 = float(q[2]);
    }
    const int per = n > 0 && n <= 32 ? 64 / n : 1;  // sub-cells per pass
    const int sub = per > 1 ? lane / n : 0;         // this lane's sub-cell of the pass
    for (int w = 0; w < words; ++w) {
        const int j = per > 1 ? lane - sub * n : w * 64 + lane;
        const bool act = j < n && sub < per;
        float c[3] = {0.0f, 0.0f, 0.0f}, cb = 1.0f, sb = 0.0f, h[3] = {0.0f, 0.0f, 0.0f};
        if (act) {
            if (j < nb) {
                const Bar<float>& b = G.bars_f[L.idx[j]];
                c[0] = b.cx; c[1] = b.cy; c[2] = b.cz;
                cb = b.cb; sb = b.sb;
                h[0] = 0.5f * b.w; h[1] = 0.5f * b.t; h[2] = 0.5f * b.h;
            } else {
                const Hole<float>& o = G.holes_f[L.idx[j]];
                c[0] = o.xc; c[1] = o.ymid; c[2] = o.zc;
                h[0] = o.r; h[1] = 0.5f * tabs(o.y2 - o.y1); h[2] = o.r;
            }
        }
        float rt[3];
        extents_in_frame(W.te, cb, sb, rt);
        for (int s0 = 0; s0 < ns; s0 += per) {
            const int s = s0 + sub;
            const float q[3] = {__shfl(q0, s & 63), __shfl(q1, s & 63), __shfl(q2, s & 63)};
            const float rq[3] = {0.0f, 0.0f, 0.0f};
            const bool pass = act && s < ns &&
                              box_meets_frustum(q, rq, W.tcf, rt, c[0], c[1], c[2], cb, sb, h[0], h[1], h[2]);
            const uint64_t bal = __ballot(pass);
            if (per > 1) {
                if (act && j == 0 && s < ns) L.sel[s] = (bal >> lane) & ((1ull << n) - 1ull);
            } else if (lane == 0) {
                L.sel[s * words + w] = bal;
            }
        }
    }
}

// The candidates of word w of sub-cell s: bars in mb, holes in mh.
template <class Lists>
__device__ __forceinline__ void sel_word(const Lists& L, int s, int words, int w, int nb, uint64_t& mb, uint64_t& mh) {
    const uint64_t m = uniform_u64(L.sel[s * words + w]);
    const int lead = nb - w * 64;  // bars in this word
    const uint64_t bars = lead >= 64 ? ~0ull : (lead <= 0 ? 0ull : (1ull << lead) - 1ull);
    mb = m & bars;
    mh = m & ~bars;
}

// Bars and holes kept for sub-cell s.
template <class Lists>
__device__ __forceinline__ void sel_count(const Lists& L, int s, int words, int nb, int& kb, int& kh) {
    kb = 0;
    kh = 0;
    for (int w = 0; w < words; ++w) {
        uint64_t mb, mh;
        sel_word(L, s, words, w, nb, mb, mh);
        kb += bit_count(mb);
        kh += bit_count(mh);
    }
}

// Sub-cells c_begin .. c_end - 1 of bar d for the tile, in blocks: narrowing
// (step 2), the records of the pairs it keeps, then the rays.  use(c, n, m)
// tests sub-cells c, c + 1, ... (at most n): it returns how many and sets m's bits
// of those to trace; f32(cell, cc, C) traces the lanes' FP32
// rays and returns the lanes whose decisions came within tolerance of a
// threshold; f64(cell, cc, C, mine) traces in FP64 the rays of the lanes with
// mine set: in the FP32 kernels those of a block's flagged rays, after its FP32
// rays (which keeps the FP64 ray's registers out of the FP32 loop), in the
// all-FP64 kernels every ray.
template <bool kExact, bool kUse, class Lists, class Use, class F32, class F64>
__device__ __forceinline__ void trace_cells(const PeLaunch& A, const Bar<double>& bd, int d, int c_begin, int c_end,
                                            const WaveSetup& W, int lane, Lists& L, int nb, int nh, Use use, F32 f32,
                                            F64 f64) {
    const PeGeom& G = A.geom;
    const int n = nb + nh, words = (n + 63) / 64;
    const int block = words > 1 ? min(kBlockCells, L.sel_cap / words) : kBlockCells;
    const uint64_t below = (1ull << lane) - 1ull;
    BarRec* const bars = (BarRec*)&L.arena[n];
    HoleRec* const holes = (HoleRec*)&L.arena[L.arena_words - (int)(sizeof(HoleRec) / 8)];
    constexpr int kBarWords = sizeof(BarRec) / 8, kHoleWords = sizeof(HoleRec) / 8;
    const int room = L.arena_words - n;
    int c = c_begin;
    while (c < c_end) {  // wave-uniform
        int ns = 0, my_cell = c + lane;
        if constexpr (kUse) {
            while (c < c_end && ns < block) {
                uint64_t m;
                const int n_tested = use(c, min(c_end - c, block - ns), m);
                for (; m; m &= m - 1, ++ns)
                    if (lane == ns) my_cell = c + __ffsll((unsigned long long)m) - 1;
                c += n_tested;
            }
        } else {
            ns = min(block, c_end - c);
            c += ns;
        }
        L.sync();  // the previous block's lists are no longer read
        select_cells(A, bd, d, my_cell, ns, W, lane, L, nb, n, words);
        L.sync();
        uint64_t flagged = 0;
        if constexpr (kExact) {
            flagged = ns == 64 ? ~0ull : (1ull << ns) - 1ull;
        } else {
            int s = 0;
            while (s < ns) {
                // the records of as many sub-cells as fit: first their pairs
                int e = s, nbr = 0, nhr = 0;
                for (; e < ns; ++e) {
                    int kb, kh;
                    sel_count(L, e, words, nb, kb, kh);
                    if ((nbr + kb) * kBarWords + (nhr + kh) * kHoleWords > room) break;
                    for (int w = 0; w < words; ++w) {
                        uint64_t mb, mh;
                        sel_word(L, e, words, w, nb, mb, mh);
                        const uint32_t tag = ((uint32_t)e << 16) | (uint32_t)(w * 64 + lane);
                        if (lane_bit(mb)) bars[nbr + bit_count(mb & below)].tag = tag;
                        if (lane_bit(mh)) holes[-(nhr + bit_count(mh & below))].tag = tag;
                        nbr += bit_count(mb);
                        nhr += bit_count(mh);
                    }
                }
                if (e == s) {  // not even one sub-cell's: its rays go to FP64
                    flagged |= 1ull << s;
                    if (lane == 0) L.redo[s] = ~0ull;
                    ++s;
                    continue;
                }
                L.sync();
                for (int i0 = 0; i0 < nbr; i0 += 64) {
                    const int i = i0 + lane;
                    const uint32_t tag = i < nbr ? bars[i].tag : 0u;
                    const int cell = __shfl(my_cell, (int)(tag >> 16) & 63);
                    if (i < nbr) {
                        const int j = tag & 0xffff, k = L.idx[j];
                        double q[3];
                        cell_point(A, bd, d, cell, q);
                        float f[6];
                        const bool fast = fast_faces(G, k, q, W.tc, W.rho, f);
                        BarRec& r = bars[i];
#pragma unroll
                        for (int m = 0; m < 6; ++m) r.face[m] = f[m];
                        r.mu = G.bars_d[k].mut;
                        r.tag = (uint32_t)j | (fast ? kFastBar : 0u);
                        r.lanes = L.arena[j];
                    }
                }
                for (int i0 = 0; i0 < nhr; i0 += 64) {
                    const int i = i0 + lane;
                    const uint32_t tag = i < nhr ? holes[-i].tag : 0u;
                    const int cell = __shfl(my_cell, (int)(tag >> 16) & 63);
                    if (i < nhr) {
                        const int j = tag & 0xffff, k = L.idx[j];
                        const Hole<double>& o = G.holes_d[k];
                        double q[3];
                        cell_point(A, bd, d, cell, q);
                        HoleRec& r = holes[-i];
                        hole_rec(o, q, r);
                        r.lanes = fabs(o.y1 - o.y2) < kCylDy ? 0ull : L.arena[j];
                        r.hole = (uint32_t)k;
                    }
                }
                L.sync();
                int ib = 0, ih = 0;
                for (; s < e; ++s) {
                    const int cell = __builtin_amdgcn_readlane(my_cell, s);
                    CellCtx cc;
                    tile_cell(A, bd, d, cell, W, lane, cc);
                    RecCands<Lists> C{&L, bars + ib, holes - ih, 0, 0};
                    sel_count(L, s, words, nb, C.nb, C.nh);
                    ib += C.nb;
                    ih += C.nh;
                    const uint64_t m = __ballot(f32(cell, cc, C));
                    if (m) {
                        flagged |= 1ull << s;
                        if (lane == 0) L.redo[s] = m;
                    }
                }
                L.sync();
            }
        }
        // FP64 rays: the candidates' positions in the place of the records
        uint16_t* const cur = (uint16_t*)bars;
        while (flagged) {
            const int s = __ffsll((unsigned long long)flagged) - 1;
            flagged &= flagged - 1;
            const int cell = __builtin_amdgcn_readlane(my_cell, s);
            CellCtx cc;
            tile_cell(A, bd, d, cell, W, lane, cc);
            ListCands<Lists> C{&L, cur, 0, 0};
            sel_count(L, s, words, nb, C.nb, C.nh);
            L.sync();
            int ib = 0, ih = C.nb;
            for (int w = 0; w < words; ++w) {
                uint64_t mb, mh;
                sel_word(L, s, words, w, nb, mb, mh);
                if (lane_bit(mb)) cur[ib + bit_count(mb & below)] = (uint16_t)(w * 64 + lane);
                if (lane_bit(mh)) cur[ih + bit_count(mh & below)] = (uint16_t)(w * 64 + lane);
                ib += bit_count(mb);
                ih += bit_count(mh);
            }
            L.sync();
            f64(cell, cc, C, W.valid && (kExact || ((L.redo[s] >> lane) & 1ull)));
        }
    }
}

// Point weights of the crystal grid scatterers (kPoints; an extension with no
// reference counterpart): the sub-cells of bar d are the grid cells, and for
// each the kernel writes the first-leg weight of its centre,
//   dv mu_c,d / (4 pi |q - p|^2) exp(-att),
// att being the PE ray's attenuation up to the point (the sub-cell's own
// chord in bar d added back), to pts[((d - bar0) n_cells + cell) V + v].
// FP64 form (the exact path and FP64 re-computations); the FP32 path forms
// the same product in FP32 (relative error ~1e-7).
__device__ __forceinline__ float point_weight(const Bar<double>& bd, int n_cells, const double aux[8]) {
    const double dv = bd.w * bd.t * bd.h / n_cells;
    return float(aux[5] * exp(-aux[4] * bd.mut) * dv * bd.muc /
                 (4.0 * 3.14159265358979323846 * aux[6]));
}

__device__ __forceinline__ float point_weight_f(const Bar<double>& bd, int n_cells, const double aux[8]) {
    const float c = float(bd.w * bd.t * bd.h / n_cells * bd.muc / (4.0 * 3.14159265358979323846));
    return float(aux[5]) * exp_neg<float>(aux[4] * bd.mut) * tdiv(c, float(aux[6]));
}

// Point weights: true when row R of A.use_rows may use the weight of grid point
// qs for a voxel of the wave's tile.  With the tile's voxel centres in the ball
// (tc, rho) and the row's sub-cell centres in its bar's bounding ball (Q, rb),
// every scattering angle at qs is at least
// angle(qs - tc, Q - qs) - asin(rho / |qs - tc|) - asin(rb / |Q - qs|); when
// its cosine is 1.1e-4 below the row's window cut, the scatter kernel's
// per-lane window test rejects every such term before it reads the weight.
__device__ __forceinline__ bool row_uses_point(const double* R, const WaveSetup& W, const double qs[3]) {
    const double c_lo = R[4];
    double u[3], b[3];
    for (int k = 0; k < 3; ++k) {
        u[k] = qs[k] - W.tc[k];
        b[k] = R[k] - qs[k];
    }
    const double L = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double B = sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
    if (c_lo <= -1.5 || !(L > W.rho * (1.0 + 1e-9) + 1e-9) || !(B > R[3] * (1.0 + 1e-9) + 1e-9)) return true;
    // the angle's and the two half-angles' sines and cosines: the difference is
    // positive when cu < cos of the half-angles' sum
    const double iL = 1.0 / L, iB = 1.0 / B;
    const double cu = (u[0] * b[0] + u[1] * b[1] + u[2] * b[2]) * (iL * iB);
    const double su = sqrt(fmax(0.0, 1.0 - cu * cu));
    const double s1 = W.rho * iL, c1 = sqrt(fmax(0.0, 1.0 - s1 * s1));
    const double s2 = R[3] * iB, c2 = sqrt(fmax(0.0, 1.0 - s2 * s2));
    const double s12 = s1 * c2 + c1 * s2, c12 = c1 * c2 - s1 * s2;
    return !(cu < c12) || !(cu * c12 + su * s12 < c_lo - 1.1e-4);
}

// The grid points c, c + 1, ... (at most n) that some row may use, as many as fit
// in the lanes with a lane per (point, row): sets m's bits, returns their number.
// (A pass per point, with three arc functions in the rows' lanes, was over half of
// the point kernel: 8 rows, 184,320 points x 1,024 voxels, 9.06 ms -> 4.03 ms.)
__device__ __forceinline__ int points_used(const PeLaunch& A, const Bar<double>& bd, int d, const WaveSetup& W,
                                           int lane, int c, int n, uint64_t& m) {
    const int sh = A.n_use_rows > 1 ? 32 - __clz(A.n_use_rows - 1) : 0;
    n = min(n, 64 >> sh);
    const int i = lane >> sh, row = lane & ((1 << sh) - 1);
    bool use = false;
    if (i < n && row < A.n_use_rows) {
        double q[3];
        cell_point(A, bd, d, c + i, q);
        use = row_uses_point(A.use_rows + 5 * row, W, q);
    }
    const uint64_t b = __ballot(use), ones = ~0ull >> (64 - (1 << sh));
    m = 0;
    for (int k = 0; k < n; ++k)
        if ((b >> (k << sh)) & ones) m |= 1ull << k;
    return n;
}

// This wave's number in a block of kWaves, in scalar registers.
template <int kWaves>
__device__ __forceinline__ int block_wave() {
    return kWaves > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
}

// Sum of the lane's accumulators over the block's waves, in wave order, with
// their compensations, through the waves' candidate lists, which are done with
// (L: this wave's; slot: 0 or 1).  Every wave comes here; the sum is the first
// one's.
template <int kWaves, class T, class Lists>
__device__ __forceinline__ double block_sum(const KahanSum<T>& acc, int wave, int lane, Lists& L, int slot) {
    double s = (double)acc.s + (double)acc.c;
    L.arena[slot * 64 + lane] = (uint64_t)__double_as_longlong(s);
    __syncthreads();
    if (wave == 0)
        for (int w = 1; w < kWaves; ++w) s += __longlong_as_double((long long)(&L)[w].arena[slot * 64 + lane]);
    return s;
}

// Work item `item` of the launch (a block index: bar, tile and, for point
// weights, slice of cells) with candidate lists L.  Returns false, having
// written nothing, when the candidates overflow L.
template <bool kExact, bool kPoints, bool kEll, int kWaves = 1, bool kFew = false, class Lists>
__device__ __forceinline__ bool pe_forward_body(const PeLaunch& A, int item, Lists& L) {
    const PeGeom& G = A.geom;
    const GeomDesc& g = G.g;
    // (masking the number in blocks of one wave too made the full-size step 0.8% slower)
    const int lane = kWaves > 1 ? threadIdx.x & 63 : threadIdx.x;
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    // point weights: cells [c_begin, c_end) of the wave's slice; PE: all cells, or
    // the wave's share of them
    const int slices = kPoints ? A.cell_slices : 1;
    const int wave = item / slices;
    const int parts = kPoints ? slices : kWaves, part = kPoints ? item % slices : block_wave<kWaves>();
    const int d = A.bar0 + wave / n_tiles;
    const int tile = wave % n_tiles;
    float* out = A.dst + (int64_t)d * g.n_vox;
    const int n_cells = A.sub[0] * A.sub[1] * A.sub[2];
    const int per = (n_cells + parts - 1) / parts;
    const int c_begin = part * per;
    const int c_end = min(n_cells, c_begin + per);
    float* pts = kPoints ? A.pts + (int64_t)(d - A.bar0) * n_cells * g.n_vox : nullptr;
    const Bar<double>& bd = G.bars_d[d];
    WaveSetup W;
    wave_setup(A, d, tile, lane, W);
    if (!(bd.mut > (double)0.01f)) {  // PESysMatGen.cu:1116, :1194
        if constexpr (kPoints) {
            if (W.valid)
                for (int c = c_begin; c < c_end; ++c) pts[(int64_t)c * g.n_vox + W.v] = 0.0f;
        } else {
            if (W.valid && part == 0) out[W.v] = 0.0f;
        }
        return true;
    }
    int nb, nh;
    if (!build_candidates<kExact, kFew>(A, d, lane, W, L, nb, nh)) return false;
    L.sync();

    using T = typename std::conditional<kExact, double, float>::type;
    KahanSum<T> acc;
    unsigned fallbacks = 0;
    // Sub-cells in the reference's loop order (z outer, then x, then y;
    // PESysMatGen.cu:1193-1197); FP32 rays whose decisions came within
    // tolerance of a threshold are not added but redone in FP64.
    auto use = [&](int c, int n, uint64_t& m) {
        if constexpr (kPoints) {
            if (A.n_use_rows > 0) {
                n = points_used(A, bd, d, W, lane, c, n, m);
                if (W.valid)
                    for (int k = 0; k < n; ++k)
                        if (!((m >> k) & 1ull)) pts[(int64_t)(c + k) * g.n_vox + W.v] = 0.0f;
                return n;
            }
        }
        m = ~0ull >> (64 - n);
        return n;
    };
    trace_cells<kExact, kPoints>(
        A, bd, d, c_begin, c_end, W, lane, L, nb, nh, use,
        [&](int cell, const CellCtx& cc, const RecCands<Lists>& C) {
            bool near = false;
            if (W.valid) {
                if constexpr (kPoints) {
                    double aux[8];
                    pe_cell_ray<float, kEll>(G, d, W.p, W.ps, cc, C, near, nullptr, aux);
                    if (!near) pts[(int64_t)cell * g.n_vox + W.v] = point_weight_f(bd, n_cells, aux);
                } else {
                    const float val = pe_cell_ray<float, kEll>(G, d, W.p, W.ps, cc, C, near);
                    if (!near) acc.add((T)val);
                }
            }
            return near;
        },
        [&](int cell, const CellCtx& cc, const ListCands<Lists>& C, bool mine) {
            if (mine) {
                bool n2 = false;
                if constexpr (kPoints) {
                    double aux[8];
                    pe_cell_ray<double, kEll>(G, d, W.p, W.ps, cc, C, n2, nullptr, aux);
                    pts[(int64_t)cell * g.n_vox + W.v] = point_weight(bd, n_cells, aux);
                } else {
                    acc.add((T)pe_cell_ray<double, kEll>(G, d, W.p, W.ps, cc, C, n2));
                }
                ++fallbacks;
            }
        });
    if constexpr (!kPoints) {
        if constexpr (kWaves > 1) {
            const double sum = block_sum<kWaves>(acc, part, lane, L, 0);
            if (W.valid && part == 0) out[W.v] = float(sum);
        } else {
            if (W.valid) out[W.v] = float(acc.value());
        }
    }
    if constexpr (!kExact) {
        unsigned tot = fallbacks;
        for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
        if (lane == 0 && tot) atomicAdd(&A.counters[0], (unsigned long long)tot);
    }
    return true;
}

// 4 waves per SIMD: 128 VGPRs (the sub-cell context and the tile ball in
// scalar registers) with 180 B of scratch a lane (spills of the set-up: 6.6e10 B of
// HBM traffic on the full-size step, 6% of its rate), and 16 one-wave blocks per CU
// within the LDS (10 KB of lists each).  The projections below likewise.
// kEll: elliptical holes (the elliptic-cylinder chord compiled in; the
// all-FP64 kernels always have it).
// kFew (few_cells): 3 waves per SIMD, with few or no spills (32 B, else 180 B); so too
// the projections.
template <bool kExact, bool kEll = kExact, bool kFew = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kFew ? 3 : 4))) void pe_forward_kernel(PeLaunch A) {
    __shared__ WaveLists L;
    const int item = xcd_item((int)blockIdx.x, (int)gridDim.x);
    if (!pe_forward_body<kExact, false, kEll, 1, kFew>(A, item, L)) spill_push(A, item, threadIdx.x);
}

// kWaves waves per work item, each with its share of the sub-cells and lists of
// its own (wide_blocks).
template <bool kExact, bool kEll, int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(4))) void pe_forward_wide_kernel(
    PeLaunch A) {
    __shared__ SharedLists L[kWaves];
    const int item = xcd_item((int)blockIdx.x, (int)gridDim.x);
    if (!pe_forward_body<kExact, false, kEll, kWaves>(A, item, L[block_wave<kWaves>()]))
        spill_push(A, item, threadIdx.x);
}

// Point weights at 3 waves per SIMD (the register cap costs no spills here;
// without it the allocation lands one register above the 3-wave limit).
template <bool kExact>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void pe_points_kernel(PeLaunch A) {
    __shared__ WaveLists L;
    const int item = xcd_item((int)blockIdx.x, (int)gridDim.x);
    if (!pe_forward_body<kExact, true, kExact>(A, item, L)) spill_push(A, item, threadIdx.x);
}

// The work items the kernel above queued (counters[2] of them), redone with
// candidate lists in global memory: wave b takes queue entries b, b + grid, ...
// and its own list slot.  The entry count is wave-uniform, so every wave ends.
template <bool kExact, bool kPoints, bool kEll = kExact>
__global__ __launch_bounds__(64) void pe_forward_spill_kernel(PeLaunch A) {
    SpillLists L = spill_lists(A.spill, (int)blockIdx.x);
    const unsigned long long n = A.counters[2];
    for (unsigned long long i = blockIdx.x; i < n; i += gridDim.x) {
        __syncthreads();  // the previous item's list reads are done
        pe_forward_body<kExact, kPoints, kEll>(A, A.spill.queue[i], L);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && n) atomicAdd(&A.counters[1], n);
}

// ---- tangent --------------------------------------------------------------------------
//
// d term of one sub-cell ray along the direction v (no counterpart in the
// reference; the derivatives of its element formula, PESysMatGen.cu:1240-1357,
// as in the adjoint): term = Omega e^-att abs,
//   d att = sum_m v_m rest_m + sum_k v_t[k] l_k + v_t[d] (l1 - l2),
//   d abs = v_t[d] mu_pe (l_a e^(-mu l_a)/mu - (1 - e^(-mu l_a))/mu^2) + v_pe[d] (1 - e^(-mu l_a))/mu,
//   d term = -term d att + Omega e^-att d abs.
// dlay, aux and tan_att as pe_cell_ray returns them.
__device__ __forceinline__ double tangent_term(const PeGeom& G, int d, const double* v, double term,
                                               const double* dlay, const double* aux, double tan_att) {
    const GeomDesc& g = G.g;
    const Bar<double>& bd = G.bars_d[d];
    const double vt = v[g.n_layers + d], vpe = v[g.n_layers + g.n_det + d];
    double datt = tan_att + vt * aux[1];
#pragma unroll
    for (int m = 0; m < kMaxLayers; ++m)
        if (m < g.n_layers) datt += v[m] * dlay[m];
    const double mut = bd.mut, la = aux[2], ea = aux[3];
    const double dabs = vt * bd.mupe * (la * ea / mut - (1.0 - ea) / (mut * mut)) + vpe * (1.0 - ea) / mut;
    return -term * datt + aux[0] * dabs;
}

// Work item `item` (bar, tile) of the tangent: as pe_forward_body, with the
// derivative summed beside the element.  Returns false, having written
// nothing, when the candidates overflow L.
template <bool kExact, int kWaves = 1, class Lists>
__device__ __forceinline__ bool pe_tangent_body(const PeLaunch& A, const PeTangent& TG, int item, Lists& L) {
    const PeGeom& G = A.geom;
    const GeomDesc& g = G.g;
    const int lane = kWaves > 1 ? threadIdx.x & 63 : threadIdx.x, part = block_wave<kWaves>();
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int d = item / n_tiles;
    const int tile = item % n_tiles;
    const int n_cells = A.sub[0] * A.sub[1] * A.sub[2];
    const Bar<double>& bd = G.bars_d[d];
    WaveSetup W;
    wave_setup(A, d, tile, lane, W);
    const int64_t o = (int64_t)d * g.n_vox + W.v;
    if (!(bd.mut > (double)0.01f)) {  // PESysMatGen.cu:1116, :1194
        if (W.valid && part == 0) {
            TG.d_out[o] = 0.0f;
            if (TG.a_out) TG.a_out[o] = 0.0f;
        }
        return true;
    }
    int nb, nh;
    if (!build_candidates<kExact, false>(A, d, lane, W, L, nb, nh)) return false;
    L.sync();
    using T = typename std::conditional<kExact, double, float>::type;
    KahanSum<T> acc;
    KahanSum<double> dacc;
    const int per = (n_cells + kWaves - 1) / kWaves, c_begin = part * per, c_end = min(n_cells, c_begin + per);
    unsigned fallbacks = 0;
    const double* vbar = TG.v + g.n_layers;
    trace_cells<kExact, false>(
        A, bd, d, c_begin, c_end, W, lane, L, nb, nh, [](int) { return true; },
        [&](int, const CellCtx& cc, const RecCands<Lists>& C) {
            bool near = false;
            if (W.valid) {
                double dlay[kMaxLayers], aux[8], tatt = 0.0;
                const float val = pe_cell_ray<float, false, true>(G, d, W.p, W.ps, cc, C, near, dlay, aux, nullptr, 0,
                                                            vbar, &tatt);
                if (!near) {
                    acc.add((T)val);
                    dacc.add(tangent_term(G, d, TG.v, (double)val, dlay, aux, tatt));
                }
            }
            return near;
        },
        [&](int, const CellCtx& cc, const ListCands<Lists>& C, bool mine) {
            if (mine) {
                bool n2 = false;
                double dlay[kMaxLayers], aux[8], tatt = 0.0;
                const double val = pe_cell_ray<double, kExact>(G, d, W.p, W.ps, cc, C, n2, dlay, aux, nullptr, 0,
                                                               vbar, &tatt);
                acc.add((T)val);
                dacc.add(tangent_term(G, d, TG.v, val, dlay, aux, tatt));
                ++fallbacks;
            }
        });
    if constexpr (kWaves > 1) {
        const double ds = block_sum<kWaves>(dacc, part, lane, L, 0);
        const double as = TG.a_out ? block_sum<kWaves>(acc, part, lane, L, 1) : 0.0;
        if (W.valid && part == 0) {
            TG.d_out[o] = float(ds);
            if (TG.a_out) TG.a_out[o] = float(as);
        }
    } else if (W.valid) {
        TG.d_out[o] = float(dacc.value());
        if (TG.a_out) TG.a_out[o] = float(acc.value());
    }
    if constexpr (!kExact) {
        unsigned tot = fallbacks;
        for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
        if (lane == 0 && tot) atomicAdd(&A.counters[0], (unsigned long long)tot);
    }
    return true;
}

template <bool kExact>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void pe_tangent_kernel(PeLaunch A, PeTangent TG) {
    __shared__ WaveLists L;
    if (!pe_tangent_body<kExact>(A, TG, (int)blockIdx.x, L)) spill_push(A, (int)blockIdx.x, threadIdx.x);
}

template <bool kExact, int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(3))) void pe_tangent_wide_kernel(
    PeLaunch A, PeTangent TG) {
    __shared__ SharedLists L[kWaves];
    if (!pe_tangent_body<kExact, kWaves>(A, TG, (int)blockIdx.x, L[block_wave<kWaves>()]))
        spill_push(A, (int)blockIdx.x, threadIdx.x);
}

template <bool kExact>
__global__ __launch_bounds__(64) void pe_tangent_spill_kernel(PeLaunch A, PeTangent TG) {
    SpillLists L = spill_lists(A.spill, (int)blockIdx.x);
    const unsigned long long n = A.counters[2];
    for (unsigned long long i = blockIdx.x; i < n; i += gridDim.x) {
        __syncthreads();
        pe_tangent_body<kExact>(A, TG, A.spill.queue[i], L);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && n) atomicAdd(&A.counters[1], n);
}

// ---- adjoint -------------------------------------------------------------------------
//
// dL/dmu of L = sum w[d][v] A[d][v].  Per sub-cell ray with term c (the
// forward contribution) and weight w (from the derivatives of the reference
// element formula, PESysMatGen.cu:1240-1357):
//   layer m:         -w c (T_m / cos(alpha) - sum of hole chords), when counted
//   bar k != d:      -w c l_k
//   mu_total of d:   -w c (l1 - l2) + w Omega e^-att mu_pe (l_a e^(-mu l_a)/mu - (1 - e^(-mu l_a))/mu^2)
//   mu_pe of d:      w Omega e^-att (1 - e^(-mu l_a)) / mu
// The chords through other bars are recomputed after the forward term, not
// stored.  One wave handles detector d and work items g, g + G, ... (an item
// is a tile, or a tile's range of sub-cells when bars x tiles alone would
// leave the GPU under-filled); partial sums
// go to a per-(d, g) row of the scratch buffer (bar mu_total partials dense
// over all bars, then the layer, mu_pe and loss slots), added in a fixed
// order, and pe_grad_reduce sums the rows in a fixed order: the result does
// not depend on scheduling.

// x moved across lanes by a DPP control (0 where the source lane is none).
template <int kCtrl, int kRows>
__device__ __forceinline__ double dpp_move(double x) {
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kCtrl, kRows, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), kCtrl, kRows, 0xf, false);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Sum over the wave, the same for every lane: shifts within the rows of 16 lanes,
// then the rows' last lanes broadcast, so that lane 63 holds the sum.  (The
// adjoint takes one per candidate and layer of every sub-cell: six rounds through
// the LDS crossbar each, gradient over 2,048 bars and 16 x 16 x 4 voxels, 8% less.)
__device__ __forceinline__ double wave_sum(double x) {
    x += dpp_move<0x111, 0xf>(x);  // row_shr:1
    x += dpp_move<0x112, 0xf>(x);  // row_shr:2
    x += dpp_move<0x114, 0xf>(x);  // row_shr:4
    x += dpp_move<0x118, 0xf>(x);  // row_shr:8
    x += dpp_move<0x142, 0xa>(x);  // row_bcast:15
    x += dpp_move<0x143, 0xc>(x);  // row_bcast:31
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), 63);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Per-wave adjoint accumulators: per-lane sums for bar d's own mu and the
// loss, wave sums (in LDS, added by lane 0 in a fixed order) for the layers
// and, per tile, for each candidate bar.
struct AdjAcc {
    double own_mut = 0.0, own_mupe = 0.0, loss = 0.0;
};

// Adjoint contributions of one sub-cell for the lanes with `active` set.  In
// FP32 a lane whose ray came within tolerance of a threshold contributes
// nothing and is reported through the return value (the caller redoes it in
// FP64).  Every lane of the wave takes part in the wave sums.
template <class T, bool kEll, class Cands>
__device__ bool adjoint_cell(const PeGeom& G, int d, int lane, const WaveSetup& W, const Cands& C,
                             const CellCtx& cc, bool active, double wv, AdjAcc& acc, double* lay_acc,
                             double* cand_acc, float* keep = nullptr) {
    const GeomDesc& g = G.g;
    const Bar<double>& bd = G.bars_d[d];
    const double mut = bd.mut, mupe = bd.mupe;
    double term = 0.0, dlay[kMaxLayers], aux[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < kMaxLayers; ++m) dlay[m] = 0.0;
    bool near = false;
    if (active) {
        term = (double)pe_cell_ray<T, kEll, true>(G, d, W.p, W.ps, cc, C, near, dlay, aux, keep, 64);
        if (kGuarded<T> && near) active = false;
    }
    const double cw = active ? wv * term : 0.0;
    if (active) {
        const double la = aux[2], ea = aux[3], effom = aux[0];
        acc.loss += cw;
        acc.own_mut += -cw * aux[1] + wv * effom * mupe * (la * ea / mut - (1.0 - ea) / (mut * mut));
        acc.own_mupe += wv * effom * (1.0 - ea) / mut;
    }
#pragma unroll
    for (int m = 0; m < kMaxLayers; ++m) {
        if (m < g.n_layers) {
            const double x = wave_sum(-cw * dlay[m]);
            if (lane == 0) lay_acc[m] += x;
        }
    }
    // chords through the other bars: kept from the ray (the first kKeepChords
    // candidates, FP32 rays) or recomputed
    double D[3], dd = 0.0, inv_dd = 0.0;
    SegDir<T> sw;
    T tol_d = T(0);
    if (!keep || C.nbars() > kKeepChords) {  // wave-uniform
        bool nd = false;
        ray_dir<T>(W.p, cc.q, D, dd, sw, tol_d, nd);
        inv_dd = 1.0 / dd;
    }
    for (int j = 0; j < C.nbars(); ++j) {
        double x = 0.0;
        if (active && cw != 0.0 && C.bar_on(j)) {
            double l;
            if (keep && j < kKeepChords) {
                l = (double)keep[j * 64];
            } else {
                bool n3 = false;
                l = (double)other_bar_chord<T>(G, C.bar(j), W.p, D, dd, inv_dd, cc.q, sw, tol_d, n3);
            }
            x = -cw * l;
        }
        x = wave_sum(x);
        if (lane == 0) cand_acc[C.pos(j)] += x;
    }
    return near;
}

// Adjoint of work item `item` (a block index: bar d, group of tiles) with
// candidate lists L and per-candidate sums cand_acc.  Returns false when the
// candidates overflow L (its scratch row is then incomplete; the spill kernel
// rewrites all of it).
template <bool kExact, class Lists>
__device__ __forceinline__ bool pe_backward_body(const PeLaunch& A, const PeGradScratch& S, int item,
                                                 Lists& L, double* cand_acc) {
    __shared__ double lay_acc[kMaxLayers];
    __shared__ float keep[kKeepChords * 64];  // FP32 rays' chords, [candidate][lane]
    const PeGeom& G = A.geom;
    const GeomDesc& g = G.g;
    const int lane = threadIdx.x;
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int d = item / S.groups;
    const int grp = item % S.groups;
    const Bar<double>& bd = G.bars_d[d];
    double* out_row = S.rows + (int64_t)item * S.stride;
    // the bars' mu_total partials accumulate in this wave's own row of the
    // scratch buffer (no other wave writes it; LDS would cap the occupancy)
    for (int k = lane; k < g.n_det; k += 64) out_row[k] = 0.0;
    if (lane < kMaxLayers) lay_acc[lane] = 0.0;
    AdjAcc acc;
    unsigned fallbacks = 0;
    bool overflow = false;
    __syncthreads();
    if (bd.mut > (double)0.01f) {
        const int n_cells = A.sub[0] * A.sub[1] * A.sub[2];
        // work items: (tile, range of sub-cells); item i is tile i / cs, range i % cs
        const int cs = S.cell_slices;
        const int per = (n_cells + cs - 1) / cs;
        for (int item = grp; item < n_tiles * cs; item += S.groups) {
            const int tile = item / cs;
            const int c_begin = (item % cs) * per, c_end = min(n_cells, c_begin + per);
            WaveSetup W;
            wave_setup(A, d, tile, lane, W);
            int nb, nh;
            if (!build_candidates<kExact, true>(A, d, lane, W, L, nb, nh)) {
                overflow = true;
                break;
            }
            for (int j = lane; j < nb; j += 64) cand_acc[j] = 0.0;
            const double wv = W.valid ? (double)S.w[(int64_t)d * g.n_vox + W.v] : 0.0;
            __syncthreads();
            trace_cells<kExact, false>(
                A, bd, d, c_begin, c_end, W, lane, L, nb, nh, [](int) { return true; },
                [&](int, const CellCtx& cc, const RecCands<Lists>& C) {
                    return adjoint_cell<float, false>(G, d, lane, W, C, cc, W.valid, wv, acc, lay_acc, cand_acc,
                                                      keep + lane);
                },
                [&](int, const CellCtx& cc, const ListCands<Lists>& C, bool mine) {
                    adjoint_cell<double, kExact>(G, d, lane, W, C, cc, mine, wv, acc, lay_acc, cand_acc);
                    fallbacks += mine;
                });
            __syncthreads();
            // fold this tile's candidate partials into the dense row (one
            // entry per candidate, each bar at most once per tile)
            for (int j = lane; j < nb; j += 64) out_row[L.idx[j]] += cand_acc[j];
            __syncthreads();
        }
    }
    const double own_mut = wave_sum(acc.own_mut);
    const double own_mupe = wave_sum(acc.own_mupe);
    const double loss = wave_sum(acc.loss);
    __syncthreads();  // the lanes' row updates before lane 0 adds to out_row[d]
    if (lane == 0) {
        out_row[d] += own_mut;
        for (int m = 0; m < g.n_layers; ++m) out_row[g.n_det + m] = lay_acc[m];
        out_row[g.n_det + g.n_layers] = own_mupe;
        out_row[g.n_det + g.n_layers + 1] = loss;
    }
    if (overflow) return false;
    if constexpr (!kExact) {
        unsigned tot = fallbacks;
        for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
        if (lane == 0 && tot) atomicAdd(&A.counters[0], (unsigned long long)tot);
    }
    return true;
}

// 3 waves per SIMD (LDS and a 168-VGPR cap).  kFew (few_cells): 2, without spills.
template <bool kExact, bool kFew = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kFew ? 2 : 3))) void pe_backward_kernel(
    PeLaunch A, PeGradScratch S) {
    __shared__ AdjointLists L;
    __shared__ double cand_acc[kCapBarsAdjoint];
    if (!pe_backward_body<kExact>(A, S, (int)blockIdx.x, L, cand_acc)) spill_push(A, (int)blockIdx.x, threadIdx.x);
}

// Queued work items of pe_backward_kernel redone with lists in global memory
// (as pe_forward_spill_kernel); each rewrites its whole scratch row.
template <bool kExact>
__global__ __launch_bounds__(64) void pe_backward_spill_kernel(PeLaunch A, PeGradScratch S) {
    SpillLists L = spill_lists(A.spill, (int)blockIdx.x);
    const unsigned long long n = A.counters[2];
    for (unsigned long long i = blockIdx.x; i < n; i += gridDim.x) {
        __syncthreads();
        pe_backward_body<kExact>(A, S, A.spill.queue[i], L, L.cand_acc);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && n) atomicAdd(&A.counters[1], n);
}

// grad[0 .. Lc-1]: layers; grad[Lc + k]: mu_total of bar k; grad[Lc + N + k]:
// mu_pe of bar k; grad[Lc + 2N]: the loss.  One block per entry, rows in a fixed order.
__global__ __launch_bounds__(256) void pe_grad_reduce(PeGradScratch S, int n_det, int n_layers,
                                                      double* grad) {
    // one block per entry: thread t sums rows t, t + 256, ... in order, then a
    // fixed tree over the threads (the same order on every run)
    __shared__ double part[256];
    const int i = blockIdx.x;
    const int t = threadIdx.x;
    const int64_t n_rows = (int64_t)n_det * S.groups;
    double s = 0.0;
    if (i < n_layers) {
        for (int64_t r = t; r < n_rows; r += 256) s += S.rows[r * S.stride + n_det + i];
    } else if (i < n_layers + n_det) {
        const int k = i - n_layers;
        for (int64_t r = t; r < n_rows; r += 256) s += S.rows[r * S.stride + k];
    } else if (i < n_layers + 2 * n_det) {
        const int k = i - n_layers - n_det;
        for (int grp = t; grp < S.groups; grp += 256)
            s += S.rows[((int64_t)k * S.groups + grp) * S.stride + n_det + n_layers];
    } else {
        for (int64_t r = t; r < n_rows; r += 256) s += S.rows[r * S.stride + n_det + n_layers + 1];
    }
    part[t] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (t < h) part[t] += part[t + h];
        __syncthreads();
    }
    if (t == 0) grad[i] = part[0];
}

// ---- matrix-free projections -----------------------------------------------------------
//
// (No counterpart in the reference, which writes the matrix.)  The element
// A[d][v] of one lane, formed as in pe_forward_kernel (same sub-cell order,
// same FP64 redo of near rays), is used at once instead of being stored:
// forward projection y[d] = sum_v A[d][v] x[v], back-projection
// x[v] = sum_d A[d][v] y[d].  Sums are FP64 in a fixed order.

// A[d][v] of this lane for bar d and the wave's tile (W set up for them) into
// a: 0 for a bar below the mu threshold.  Returns false (wave-uniform) when
// the candidates overflow L; adds the lane's FP64 re-computations to fallbacks.
template <bool kExact, bool kEll, bool kFew, class Lists>
__device__ bool pe_element(const PeLaunch& A, int d, int lane, const WaveSetup& W, Lists& L,
                           unsigned& fallbacks, double& a) {
    const PeGeom& G = A.geom;
    const Bar<double>& bd = G.bars_d[d];
    a = 0.0;
    if (!(bd.mut > (double)0.01f)) return true;  // PESysMatGen.cu:1116, :1194
    int nb, nh;
    __syncthreads();  // the lists of the previous element are no longer read
    if (!build_candidates<kExact, kFew>(A, d, lane, W, L, nb, nh)) return false;
    __syncthreads();
    using T = typename std::conditional<kExact, double, float>::type;
    KahanSum<T> acc;
    trace_cells<kExact, false>(
        A, bd, d, 0, A.sub[0] * A.sub[1] * A.sub[2], W, lane, L, nb, nh, [](int) { return true; },
        [&](int, const CellCtx& cc, const RecCands<Lists>& C) {
            bool near = false;
            if (W.valid) {
                const float val = pe_cell_ray<float, kEll>(G, d, W.p, W.ps, cc, C, near);
                if (!near) acc.add((T)val);
            }
            return near;
        },
        [&](int, const CellCtx& cc, const ListCands<Lists>& C, bool mine) {
            if (mine) {
                bool n2 = false;
                acc.add((T)pe_cell_ray<double, kEll>(G, d, W.p, W.ps, cc, C, n2));
                ++fallbacks;
            }
        });
    // the element as the matrix kernel stores it (FP32), so that projecting equals
    // multiplying by the stored matrix; wide blocks (wide_blocks) add their waves'
    // compensated sums in FP64, which rounds to the same float unless the sum lies
    // within its last bits of a tie (none of 1e7 sums tried)
    a = (double)float(acc.value());
    return true;
}

__device__ __forceinline__ void add_fallbacks(const PeLaunch& A, int lane, unsigned fallbacks) {
    unsigned tot = fallbacks;
    for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
    if (lane == 0 && tot) atomicAdd(&A.counters[0], (unsigned long long)tot);
}

// Forward projection of work item `item` (bar d, voxel tile): the wave's share
// of y[d] goes to partial[item].  Returns false, having written nothing, when
// the candidates overflow L.
template <bool kExact, bool kEll, bool kFew = false, class Lists>
__device__ __forceinline__ bool pe_project_body(const PeLaunch& A, const float* x, double* partial, int item,
                                                Lists& L) {
    const int lane = threadIdx.x;
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int d = item / n_tiles;
    const int tile = item % n_tiles;
    WaveSetup W;
    wave_setup(A, d, tile, lane, W);
    unsigned fallbacks = 0;
    double a;
    if (!pe_element<kExact, kEll, kFew>(A, d, lane, W, L, fallbacks, a)) return false;
    const double s = wave_sum(W.valid ? a * (double)x[W.v] : 0.0);
    if (lane == 0) partial[item] = s;
    if constexpr (!kExact) add_fallbacks(A, lane, fallbacks);
    return true;
}

template <bool kExact, bool kEll = kExact, bool kFew = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kFew ? 3 : 4))) void pe_project_kernel(PeLaunch A, const float* x, double* partial) {
    __shared__ WaveLists L;
    if (!pe_project_body<kExact, kEll, kFew>(A, x, partial, (int)blockIdx.x, L)) spill_push(A, (int)blockIdx.x, threadIdx.x);
}

// Back-projection of work item `item` (group of `group` consecutive bars,
// voxel tile), looping over the group's bars (those with y[d] = 0 skipped);
// each lane's share of x[v] goes to partial[group][v].  Returns false, having
// written nothing, when the candidates of one of the bars overflow L.
template <bool kExact, bool kEll, bool kFew = false, class Lists>
__device__ __forceinline__ bool pe_backproject_body(const PeLaunch& A, const float* y, int group,
                                                    double* partial, int item, Lists& L) {
    const GeomDesc& g = A.geom.g;
    const int lane = threadIdx.x;
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int grp = item / n_tiles;
    const int tile = item % n_tiles;
    const int d0 = grp * group, d1 = min(g.n_det, d0 + group);
    unsigned fallbacks = 0;
    double acc = 0.0;
    for (int d = d0; d < d1; ++d) {
        const float yd = y[d];
        if (yd == 0.0f) continue;  // wave-uniform
        WaveSetup W;
        wave_setup(A, d, tile, lane, W);
        double a;
        if (!pe_element<kExact, kEll, kFew>(A, d, lane, W, L, fallbacks, a)) return false;
        acc += a * (double)yd;
    }
    // the lane's voxel (it does not depend on the bar)
    const int t0 = tile % A.tiles[0], t1 = (tile / A.tiles[0]) % A.tiles[1],
              t2 = tile / (A.tiles[0] * A.tiles[1]);
    const int ix = t0 * A.tile[0] + lane % A.tile[0];
    const int iy = t1 * A.tile[1] + (lane / A.tile[0]) % A.tile[1];
    const int iz = t2 * A.tile[2] + lane / (A.tile[0] * A.tile[1]);
    if (ix < g.nx && iy < g.ny && iz < g.nz)
        partial[(int64_t)grp * g.n_vox + ix + (int64_t)iy * g.nx + (int64_t)iz * g.nx * g.ny] = acc;
    if constexpr (!kExact) add_fallbacks(A, lane, fallbacks);
    return true;
}

template <bool kExact, bool kEll = kExact, bool kFew = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kFew ? 3 : 4))) void pe_backproject_kernel(
    PeLaunch A, const float* y, int group, double* partial) {
    __shared__ WaveLists L;
    if (!pe_backproject_body<kExact, kEll, kFew>(A, y, group, partial, (int)blockIdx.x, L)) spill_push(A, (int)blockIdx.x, threadIdx.x);
}

// Queued work items of the projection kernels redone with lists in global
// memory (as pe_forward_spill_kernel).
template <bool kExact, bool kBack, bool kEll = kExact>
__global__ __launch_bounds__(64) void pe_project_spill_kernel(PeLaunch A, const float* in, int group,
                                                              double* partial) {
    SpillLists L = spill_lists(A.spill, (int)blockIdx.x);
    const unsigned long long n = A.counters[2];
    for (unsigned long long i = blockIdx.x; i < n; i += gridDim.x) {
        __syncthreads();
        if constexpr (kBack)
            pe_backproject_body<kExact, kEll>(A, in, group, partial, A.spill.queue[i], L);
        else
            pe_project_body<kExact, kEll>(A, in, partial, A.spill.queue[i], L);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && n) atomicAdd(&A.counters[1], n);
}

// out[i] = sum_k partial[k * stride + i * step] for k < n, in k order.
__global__ __launch_bounds__(256) void sum_rows_kernel(const double* partial, int64_t n_out, int n,
                                                       int64_t stride, int64_t step, float* out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_out) return;
    KahanSum<double> s;
    for (int k = 0; k < n; ++k) s.add(partial[(int64_t)k * stride + i * step]);
    out[i] = float(s.value());
}

}  // namespace

namespace {

// Checks the spill area against a launch of `blocks` blocks, clears the
// launch's queue length, and returns the spill kernel's grid.  A launch with
// no spill area (queue == nullptr; the caller has cleared counters[2]) gets
// grid 0: its overflowing work items are only counted in counters[2].
hipError_t spill_begin(const PeLaunch& A, int64_t blocks, hipStream_t stream, unsigned& spill_grid) {
    const PeSpill& S = A.spill;
    spill_grid = 0;
    if (!S.queue) return hipSuccess;
    if (!S.slots || S.n_slots < 1 || blocks > S.queue_cap || S.cap_bars < A.geom.g.n_det ||
        S.cap_holes < A.geom.g.n_holes || S.slot_bytes < pe_spill_slot_bytes(S.cap_bars, S.cap_holes))
        return hipErrorInvalidValue;
    spill_grid = (unsigned)std::min<int64_t>(S.n_slots, blocks);
    return hipMemsetAsync(A.counters + 2, 0, sizeof(unsigned long long), stream);
}

}  // namespace

// Blocks whose waves share an item's sub-cells (4 waves, or the 3 that the
// tangent's registers let a SIMD hold), where one wave per item is at most two per
// SIMD: bound by latency then, 1,024 items of 64 sub-cells 197 -> 117 us a call
// (tangent kernel 217 -> 147 us), 2,048 items 306 -> 249 us (tangent 317 -> 271).
// From 4,096 items on the waves' own candidate lists cost more than they gain (467
// -> 486 us), and below 16 sub-cells there is little to share (16: 159 -> 112 us).
// The count is of the whole detector: a range of its rows is summed alike.
constexpr int kWideWaves = 4, kTangentWaves = 3;
static void launch_forward_wide(const PeLaunch& A, bool exact, int64_t blocks, hipStream_t stream);
static void launch_tangent_wide(const PeLaunch& A, const PeTangent& TG, bool exact, int64_t blocks, hipStream_t stream);
static bool wide_blocks(const PeLaunch& A) {
    const int64_t items = (int64_t)A.geom.g.n_det * A.tiles[0] * A.tiles[1] * A.tiles[2];
    return items <= 2048 && A.sub[0] * A.sub[1] * A.sub[2] >= 4 * kWideWaves;
}

// FP32 launches of few sub-cells over small tiles: setting a wave up (its lists, the
// first block of sub-cells) is then most of its work, and registers spilled there
// cost more than a wave more per SIMD gives.  2,048 bars, 8,192 voxels of 0.6 mm, one
// sub-cell: matrix 2.11 -> 1.76 ms (1.97 with one sub-cell narrowed at a time), panel
// turned by 0.25 rad 3.00 -> 2.45 (2.47; 4 sub-cells 4.57 -> 4.13), adjoint kernel of
// 1,024 voxels 0.65 -> 0.51 (0.58); 64 turned bars, 10,752 voxels of 0.3 mm, 6
// sub-cells 156 -> 130 us (141).  With more sub-cells or wider tiles, whose candidate
// lists are longer, the rays count: 2,048 bars, 8 sub-cells, half diagonal of a tile
// 1.6 mm 2.35 and 2.33 ms, 2.6 mm 2.65 and 2.70; 4 sub-cells, 5.2 mm 6.0 and 6.4; one,
// 10.4 mm 14.9 and 16.9.  The kernels with the elliptic chord spill more and gain up to
// twice that (512 bars, 8 sub-cells, 2.6 mm 899 -> 821 us, 6.5 mm 1.50 ms both).
// (Both sides have since gained from frustum_cut and append_candidates alike: matrix
// and turned panel 1.60 and 2.27 ms.)
static bool few_cells(const PeLaunch& A) {
    const GeomDesc& g = A.geom.g;
    const double x = (A.tile[0] - 1) * g.wx, y = (A.tile[1] - 1) * g.wy, z = (A.tile[2] - 1) * g.wz;
    const double rho = 0.5 * std::sqrt(x * x + y * y + z * z);
    const int cells = A.sub[0] * A.sub[1] * A.sub[2];
    return cells <= 8 && rho <= 5.0 && cells * rho <= (A.ell ? 40.0 : 20.0);
}

hipError_t launch_pe_tangent(const PeLaunch& A, const PeTangent& TG, bool exact, hipStream_t stream) {
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int64_t blocks = (int64_t)n_tiles * A.geom.g.n_det;
    if (blocks <= 0) return hipSuccess;
    unsigned sg = 0;
    hipError_t e = spill_begin(A, blocks, stream, sg);
    if (e != hipSuccess) return e;
    const bool wide = wide_blocks(A);
    if (exact) {
        if (wide)
            launch_tangent_wide(A, TG, exact, blocks, stream);
        else
            hipLaunchKernelGGL(pe_tangent_kernel<true>, dim3((unsigned)blocks), dim3(64), 0, stream, A, TG);
        if (sg) hipLaunchKernelGGL(pe_tangent_spill_kernel<true>, dim3(sg), dim3(64), 0, stream, A, TG);
    } else {
        if (wide)
            launch_tangent_wide(A, TG, exact, blocks, stream);
        else
            hipLaunchKernelGGL(pe_tangent_kernel<false>, dim3((unsigned)blocks), dim3(64), 0, stream, A, TG);
        if (sg) hipLaunchKernelGGL(pe_tangent_spill_kernel<false>, dim3(sg), dim3(64), 0, stream, A, TG);
    }
    return hipGetLastError();
}

hipError_t launch_pe_backward(const PeLaunch& A, const PeGradScratch& S, bool exact, double* grad,
                              hipStream_t stream) {
    const int64_t blocks = (int64_t)A.geom.g.n_det * S.groups;
    if (blocks <= 0) return hipSuccess;
    unsigned sg = 0;
    hipError_t e = spill_begin(A, blocks, stream, sg);
    if (e != hipSuccess) return e;
    if (exact) {
        hipLaunchKernelGGL(pe_backward_kernel<true>, dim3((unsigned)blocks), dim3(64), 0, stream, A, S);
        if (sg) hipLaunchKernelGGL(pe_backward_spill_kernel<true>, dim3(sg), dim3(64), 0, stream, A, S);
    } else {
        if (few_cells(A))
            hipLaunchKernelGGL((pe_backward_kernel<false, true>), dim3((unsigned)blocks), dim3(64), 0, stream, A, S);
        else
            hipLaunchKernelGGL(pe_backward_kernel<false>, dim3((unsigned)blocks), dim3(64), 0, stream, A, S);
        if (sg) hipLaunchKernelGGL(pe_backward_spill_kernel<false>, dim3(sg), dim3(64), 0, stream, A, S);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int n_out = A.geom.g.n_layers + 2 * A.geom.g.n_det + 1;
    hipLaunchKernelGGL(pe_grad_reduce, dim3(n_out), dim3(256), 0, stream, S, A.geom.g.n_det,
                       A.geom.g.n_layers, grad);
    return hipGetLastError();
}

namespace {

// One thread per (bar, sub-cell): the sub-cell context the PE kernels would
// form with make_cell_ctx_linear (same code, same values).
__global__ __launch_bounds__(256) void cell_table_kernel(PeGeom G, int bar0, int n_bars, int s0, int s1,
                                                         int s2, CellCtx* out) {
    const int n_cells = s0 * s1 * s2;
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= (int64_t)n_bars * n_cells) return;
    const int b = (int)(tid / n_cells), cell = (int)(tid % n_cells);
    const int sub[3] = {s0, s1, s2};
    CellCtx cc;
    make_cell_ctx_linear(G.bars_d[bar0 + b], cell, sub, cc);
    cc.gate_clear = 0;
    out[tid] = cc;
}

}  // namespace

hipError_t launch_cell_table(const PeGeom& geom, int bar0, int n_bars, const int sub[3], CellCtx* out,
                             hipStream_t stream) {
    const int64_t total = (int64_t)n_bars * sub[0] * sub[1] * sub[2];
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(cell_table_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream,
                       geom, bar0, n_bars, sub[0], sub[1], sub[2], out);
    return hipGetLastError();
}

hipError_t launch_pe_forward(const PeLaunch& A, bool exact, hipStream_t stream) {
    return launch_pe_forward_rows(A, exact, 0, A.geom.g.n_det, stream);
}

hipError_t launch_pe_forward_rows(const PeLaunch& A, bool exact, int bar0, int n_bars, hipStream_t stream) {
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    if (bar0 < 0 || n_bars < 0 || bar0 + n_bars > A.geom.g.n_det) return hipErrorInvalidValue;
    const int64_t blocks = (int64_t)n_tiles * n_bars;
    if (blocks <= 0) return hipSuccess;
    PeLaunch B = A;
    B.bar0 = bar0;
    B.cell_slices = 1;
    unsigned sg = 0;
    hipError_t e = spill_begin(B, blocks, stream, sg);
    if (e != hipSuccess) return e;
    const bool wide = wide_blocks(A), few = few_cells(A);
    const dim3 grid((unsigned)blocks), threads(64);
    if (exact) {
        if (wide)
            launch_forward_wide(B, exact, blocks, stream);
        else
            hipLaunchKernelGGL(pe_forward_kernel<true>, grid, threads, 0, stream, B);
        if (sg) hipLaunchKernelGGL((pe_forward_spill_kernel<true, false>), dim3(sg), dim3(64), 0, stream, B);
    } else if (A.ell) {
        if (wide)
            launch_forward_wide(B, exact, blocks, stream);
        else
            hipLaunchKernelGGL((few ? pe_forward_kernel<false, true, true> : pe_forward_kernel<false, true>), grid,
                               threads, 0, stream, B);
        if (sg)
            hipLaunchKernelGGL((pe_forward_spill_kernel<false, false, true>), dim3(sg), dim3(64), 0, stream, B);
    } else {
        if (wide)
            launch_forward_wide(B, exact, blocks, stream);
        else
            hipLaunchKernelGGL((few ? pe_forward_kernel<false, false, true> : pe_forward_kernel<false>), grid, threads, 0,
                               stream, B);
        if (sg) hipLaunchKernelGGL((pe_forward_spill_kernel<false, false>), dim3(sg), dim3(64), 0, stream, B);
    }
    return hipGetLastError();
}

hipError_t launch_pe_points(const PeLaunch& A, bool exact, int bar0, int n_bars, hipStream_t stream) {
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int n_cells = A.sub[0] * A.sub[1] * A.sub[2];
    const int64_t waves = (int64_t)n_tiles * n_bars;
    if (waves <= 0) return hipSuccess;
    PeLaunch B = A;
    B.bar0 = bar0;
    // cells split over waves until the launch holds about 32768 waves, with
    // at least 64 cells per wave (each wave builds its own candidate lists)
    int64_t slices = (32768 + waves - 1) / waves;
    slices = std::min<int64_t>(slices, std::max(1, n_cells / 64));
    B.cell_slices = (int)std::max<int64_t>(slices, 1);
    const int64_t blocks = waves * B.cell_slices;
    unsigned sg = 0;
    hipError_t e = spill_begin(B, blocks, stream, sg);
    if (e != hipSuccess) return e;
    if (exact) {
        hipLaunchKernelGGL(pe_points_kernel<true>, dim3((unsigned)blocks), dim3(64), 0, stream, B);
        if (sg) hipLaunchKernelGGL((pe_forward_spill_kernel<true, true>), dim3(sg), dim3(64), 0, stream, B);
    } else {
        hipLaunchKernelGGL(pe_points_kernel<false>, dim3((unsigned)blocks), dim3(64), 0, stream, B);
        if (sg) hipLaunchKernelGGL((pe_forward_spill_kernel<false, true>), dim3(sg), dim3(64), 0, stream, B);
    }
    return hipGetLastError();
}

int backproject_group(const PeLaunch& A) {
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int64_t waves = (int64_t)A.geom.g.n_det * n_tiles;
    // enough waves to fill the GPU (~32768), at most 64 bars per wave
    return (int)std::min<int64_t>(64, std::max<int64_t>(1, waves / 32768));
}

size_t project_scratch(const PeLaunch& A, bool back) {
    const GeomDesc& g = A.geom.g;
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    if (!back) return (size_t)g.n_det * (size_t)n_tiles;
    const int grp = backproject_group(A);
    return (size_t)((g.n_det + grp - 1) / grp) * (size_t)g.n_vox;
}

hipError_t launch_pe_project(const PeLaunch& A, bool exact, const float* x, double* partial, float* y,
                             hipStream_t stream) {
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int64_t blocks = (int64_t)A.geom.g.n_det * n_tiles;
    if (blocks <= 0) return hipSuccess;
    unsigned sg = 0;
    hipError_t e = spill_begin(A, blocks, stream, sg);
    if (e != hipSuccess) return e;
    const bool few = few_cells(A);
    if (exact) {
        hipLaunchKernelGGL(pe_project_kernel<true>, dim3((unsigned)blocks), dim3(64), 0, stream, A, x, partial);
        if (sg) hipLaunchKernelGGL((pe_project_spill_kernel<true, false>), dim3(sg), dim3(64), 0, stream, A, x, 0,
                           partial);
    } else if (A.ell) {
        hipLaunchKernelGGL((few ? pe_project_kernel<false, true, true> : pe_project_kernel<false, true>),
                           dim3((unsigned)blocks), dim3(64), 0, stream, A, x, partial);
        if (sg)
            hipLaunchKernelGGL((pe_project_spill_kernel<false, false, true>), dim3(sg), dim3(64), 0, stream, A, x,
                               0, partial);
    } else {
        hipLaunchKernelGGL((few ? pe_project_kernel<false, false, true> : pe_project_kernel<false>),
                           dim3((unsigned)blocks), dim3(64), 0, stream, A, x, partial);
        if (sg) hipLaunchKernelGGL((pe_project_spill_kernel<false, false>), dim3(sg), dim3(64), 0, stream, A, x, 0,
                           partial);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t n = A.geom.g.n_det;  // y[d] = sum over tiles of partial[d * n_tiles + t]
    hipLaunchKernelGGL(sum_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, partial,
                       n, n_tiles, (int64_t)1, (int64_t)n_tiles, y);
    return hipGetLastError();
}

hipError_t launch_pe_backproject(const PeLaunch& A, bool exact, const float* y, double* partial, float* x,
                                 hipStream_t stream) {
    const GeomDesc& g = A.geom.g;
    const int n_tiles = A.tiles[0] * A.tiles[1] * A.tiles[2];
    const int grp = backproject_group(A);
    const int n_grp = (g.n_det + grp - 1) / grp;
    const int64_t blocks = (int64_t)n_grp * n_tiles;
    if (blocks <= 0) return hipSuccess;
    unsigned sg = 0;
    hipError_t e = spill_begin(A, blocks, stream, sg);
    if (e != hipSuccess) return e;
    const bool few = few_cells(A);
    if (exact) {
        hipLaunchKernelGGL(pe_backproject_kernel<true>, dim3((unsigned)blocks), dim3(64), 0, stream, A, y, grp,
                           partial);
        if (sg) hipLaunchKernelGGL((pe_project_spill_kernel<true, true>), dim3(sg), dim3(64), 0, stream, A, y, grp,
                           partial);
    } else if (A.ell) {
        hipLaunchKernelGGL((few ? pe_backproject_kernel<false, true, true> : pe_backproject_kernel<false, true>),
                           dim3((unsigned)blocks), dim3(64), 0, stream, A, y, grp, partial);
        if (sg)
            hipLaunchKernelGGL((pe_project_spill_kernel<false, true, true>), dim3(sg), dim3(64), 0, stream, A, y,
                               grp, partial);
    } else {
        hipLaunchKernelGGL((few ? pe_backproject_kernel<false, false, true> : pe_backproject_kernel<false>),
                           dim3((unsigned)blocks), dim3(64), 0, stream, A, y, grp, partial);
        if (sg) hipLaunchKernelGGL((pe_project_spill_kernel<false, true>), dim3(sg), dim3(64), 0, stream, A, y, grp,
                           partial);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t n = g.n_vox;  // x[v] = sum over groups of partial[k * V + v]
    hipLaunchKernelGGL(sum_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, partial,
                       n, n_grp, n, (int64_t)1, x);
    return hipGetLastError();
}

static void launch_forward_wide(const PeLaunch& A, bool exact, int64_t blocks, hipStream_t stream) {
    const dim3 grid((unsigned)blocks), threads(64 * kWideWaves);
    if (exact)
        hipLaunchKernelGGL((pe_forward_wide_kernel<true, true, kWideWaves>), grid, threads, 0, stream, A);
    else if (A.ell)
        hipLaunchKernelGGL((pe_forward_wide_kernel<false, true, kWideWaves>), grid, threads, 0, stream, A);
    else
        hipLaunchKernelGGL((pe_forward_wide_kernel<false, false, kWideWaves>), grid, threads, 0, stream, A);
}

static void launch_tangent_wide(const PeLaunch& A, const PeTangent& TG, bool exact, int64_t blocks,
                                hipStream_t stream) {
    const dim3 grid((unsigned)blocks), threads(64 * kTangentWaves);
    if (exact)
        hipLaunchKernelGGL((pe_tangent_wide_kernel<true, kTangentWaves>), grid, threads, 0, stream, A, TG);
    else
        hipLaunchKernelGGL((pe_tangent_wide_kernel<false, kTangentWaves>), grid, threads, 0, stream, A, TG);
}

}  // namespace smg
