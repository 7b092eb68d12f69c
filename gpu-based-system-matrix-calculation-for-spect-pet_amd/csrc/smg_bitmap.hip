// Geometry bitmaps of the scatter kernels, gfx950.
//
// The reference runs one thread per bit and sets bits with atomicOr
// (scatter.cu:1538).  Here a wave owns 64 consecutive bars k (one per lane) and
// kBmI = 4 origins i (bars, or layer-0 holes), and walks a slice of the bars j:
// the directions i -> k stay in registers, the direction j -> k is loaded once
// for the 4 rows (i, j), and what depends on (i, j) alone comes through the
// scalar unit.  A bit is then 5 FP32 operations per end of the pair (bm_margin)
// and two comparisons whose masks are the words; decisions within their rounding
// bound are redone with the reference formula in FP64.  32 rows' words are
// gathered in the lanes and stored together.
//
// The directions are a table built first, in FP64, one entry per (origin, bar):
// N^2 entries serve N^3 / 2 bits.  Bound by vector issue (~15 instructions a
// bit).  2,048 bars, crystal (4.3e9 bits, 537 MB), call with the copy out:
// 7.66 -> 2.32 ms; one lane per bit with both directions formed for each bit issued
// ~67.  6,000 bars: 184 -> 74 ms.
#include <hip/hip_runtime.h>

#include "smg_bitmap_body.hpp"
#include "smg_kernels.hpp"

// lane `at` of x becomes the wave-uniform v (v_writelane_b32)
extern "C" __device__ int smg_writelane(int v, int at, int x) __asm("llvm.amdgcn.writelane.i32");

namespace smg {

namespace {

constexpr int kBmI = 4;  // origins per wave
constexpr int kBmJ = 8;  // bars j per store: 4 x 8 rows x 2 words fill the lanes

// The rows' terms (BmRow) of kBmI origins against one bar.
struct BmRows {
    float x2[kBmI], y2[kBmI], z2[kBmI], c[kBmI], cr[kBmI];
};

// One chunk of a bitmap: origins [i0, i0 + ni) against bars [k0, k0 + nk).
struct BmChunk {
    const Sphere<double>* bars;
    const Sphere<double>* origins;  // bars (crystal) or holes (collimator)
    BmDir* dirs;                    // [origin][nk_pad]: every bar, or the chunk's holes
    BmRows* rows;                   // [block of origins][bar j]
    uint32_t* words;
    int n, i0, ni, k0, nk, nk_pad, slice;
};

template <bool kColl>
__global__ __launch_bounds__(256) void bitmap_dirs_kernel(BmChunk C) {
    const int64_t n_org = kColl ? C.ni : C.n;
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (x >= n_org * C.nk_pad) return;
    const int o = (int)(x / C.nk_pad), k = (int)(x - (int64_t)o * C.nk_pad);
    BmDir d{0.0f, 0.0f, 0.0f, 0.0f};
    if (k < C.nk) d = bm_dir(C.origins[kColl ? C.i0 + o : o], C.bars[C.k0 + k]);
    C.dirs[x] = d;
}

__global__ __launch_bounds__(256) void bitmap_rows_kernel(BmChunk C) {
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t blocks = (C.ni + kBmI - 1) / kBmI;
    if (x >= blocks * C.n * kBmI) return;
    const int64_t bj = x / kBmI;
    const int ii = (int)(x - bj * kBmI);
    const int64_t ib = bj / C.n;
    const int j = (int)(bj - ib * C.n);
    const int64_t i = ib * kBmI + ii;
    BmRow r{};
    if (i < C.ni) r = bm_row(C.origins[C.i0 + i], C.bars[j]);
    BmRows& R = C.rows[bj];
    R.x2[ii] = r.x2;
    R.y2[ii] = r.y2;
    R.z2[ii] = r.z2;
    R.c[ii] = r.c;
    R.cr[ii] = r.cr;
}

__global__ __launch_bounds__(256) void bitmap_clear_kernel(uint32_t* words, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < n; w += stride) words[w] = 0;
}

template <bool kColl, bool kWhole>
__global__ __launch_bounds__(256) void bitmap_kernel(BmChunk C) {
    const int lane = threadIdx.x & 63;
    const int run = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (run * 64 >= C.nk) return;
    const int k0 = C.k0 + run * 64, k_end = C.k0 + C.nk;
    const int ib = blockIdx.y, i0 = C.i0 + ib * kBmI, i1 = C.i0 + C.ni;
    const int jhi = min(C.n, ((int)blockIdx.z + 1) * C.slice);
    int jlo = (int)blockIdx.z * C.slice;
    if (!kColl && jlo < i0) jlo = i0;  // rows (i, j) with j < i do not exist
    if (jlo >= jhi) return;
    const BmDir* dirs = C.dirs + run * 64 + lane;
    BmDir Ui[kBmI];
#pragma unroll
    for (int ii = 0; ii < kBmI; ++ii) {
        const int i = min(i0 + ii, i1 - 1);
        Ui[ii] = dirs[(int64_t)(kColl ? i - C.i0 : i) * C.nk_pad];
    }
    typedef const __attribute__((address_space(4))) BmRows ScalarRows;
    const int64_t n = C.n;
    for (int jb = jlo; jb < jhi; jb += kBmJ) {
        int word = 0;         // lane: half (lane & 1) of row (i, j)
        float close = 1.0f;   // smallest |t|
#pragma unroll
        for (int jj = 0; jj < kBmJ; ++jj) {
            const int j = min(jb + jj, jhi - 1);
            ScalarRows* r = (ScalarRows*)(C.rows + ib * n + j);
            BmDir Uj{};
            if (!kColl) Uj = dirs[(int64_t)j * C.nk_pad];
#pragma unroll
            for (int ii = 0; ii < kBmI; ++ii) {
                float t = bm_margin(Ui[ii], r->x2[ii], r->y2[ii], r->z2[ii], r->c[ii]);
                if (!kColl) t = fmaxf(t, bm_margin(Uj, -r->x2[ii], -r->y2[ii], -r->z2[ii], r->cr[ii]));
                close = fminf(close, tabs(t));
                const uint64_t m = __ballot(t > 0.0f);
                const int at = (jj * kBmI + ii) * 2;
                word = smg_writelane((int)(uint32_t)m, at, word);
                word = smg_writelane((int)(uint32_t)(m >> 32), at + 1, word);
            }
        }
        if (__ballot(close <= kBmTol)) {  // rare: the close decisions again, in FP64
#pragma unroll 1
            for (int r = 0; r < kBmI * kBmJ; ++r) {
                const int i = i0 + r % kBmI, j = jb + r / kBmI, k = k0 + lane;
                if (i >= i1 || j >= jhi || (!kColl && i >= j)) continue;  // wave-uniform
                const BmRows& R = C.rows[ib * n + j];
                const int ii = r % kBmI;
                float t = bm_margin(dirs[(int64_t)(kColl ? i - C.i0 : i) * C.nk_pad], R.x2[ii], R.y2[ii], R.z2[ii], R.c[ii]);
                if (!kColl)
                    t = fmaxf(t, bm_margin(dirs[(int64_t)j * C.nk_pad], -R.x2[ii], -R.y2[ii], -R.z2[ii], R.cr[ii]));
                bool bit = t > 0.0f, nn = false;
                if (tabs(t) <= kBmTol && k < k_end) {
                    const Sphere<double>&I = C.origins[i], &J = C.bars[j], &K = C.bars[k];
                    bit = kColl ? bm_seen_from<double>(I, J, K, nn) : bm_crystal_pred<double>(I, J, K, nn);
                }
                const uint64_t m = __ballot(bit);
                if (lane >> 1 == r) word = (int)(uint32_t)(lane & 1 ? m >> 32 : m);
            }
        }
        const int i = i0 + ((lane / 2) % kBmI), j = jb + lane / 2 / kBmI, kx = k0 + 32 * (lane & 1);
        if (i >= i1 || j >= jhi || kx >= k_end || (!kColl && j < i)) continue;
        uint32_t w = (uint32_t)word & (~0u >> (32 - min(32, k_end - kx)));
        if (!kColl) {  // no bar lies between itself and another
            if (i == j) w = 0u;
            if ((unsigned)(i - kx) < 32u) w &= ~(1u << (i - kx));
            if ((unsigned)(j - kx) < 32u) w &= ~(1u << (j - kx));
        }
        const int64_t b = (kColl ? i * n + j : bm_row_start(i, n) + j - i) * n + kx;
        uint32_t* to = C.words + (b >> 5);
        if (kWhole) {
            *to = w;
        } else if (w) {  // rows share words: into the cleared bitmap
            const int sh = (int)(b & 31);
            const uint32_t hi = sh ? w >> (32 - sh) : 0u;
            atomicOr(to, w << sh);
            if (hi) atomicOr(to + 1, hi);
        }
    }
}

template <bool kColl>
void launch_chunk(const BmChunk& C, bool whole, hipStream_t stream) {
    const int runs = (C.nk + 63) / 64, blocks = (C.ni + kBmI - 1) / kBmI;
    const dim3 grid((unsigned)((runs + 3) / 4), (unsigned)blocks, (unsigned)((C.n + C.slice - 1) / C.slice));
    if (whole)
        hipLaunchKernelGGL((bitmap_kernel<kColl, true>), grid, dim3(256), 0, stream, C);
    else
        hipLaunchKernelGGL((bitmap_kernel<kColl, false>), grid, dim3(256), 0, stream, C);
}

// Small bitmaps, in one launch without tables: a wave owns 64 consecutive words; at
// step s lane l evaluates bit 64 s + l, and a ballot gives words 2s and 2s + 1.  A
// lane keeps its row's terms until its k wraps into the next row.
constexpr int kWordsPerRun = 64;                // one word per lane
constexpr int64_t kBitsPerRun = 32 * kWordsPerRun;

template <bool kColl>
__global__ __launch_bounds__(256) void bitmap_walk_kernel(BitmapLaunch A) {
    const int lane = threadIdx.x & 63;
    const int64_t n = A.n_det;
    const int64_t total = bm_total_bits(kColl, n, A.n_holes);
    const int64_t n_runs = (A.n_words + kWordsPerRun - 1) / kWordsPerRun;
    const int64_t stride = ((int64_t)gridDim.x * blockDim.x) >> 6;
    // the run index is the same for the 64 lanes of a wave, so every ballot
    // below sees the whole wave
    for (int64_t run = (((int64_t)blockIdx.x * blockDim.x) + threadIdx.x) >> 6; run < n_runs;
         run += stride) {
        int64_t b = run * kBitsPerRun + lane;
        BitRow r{};
        int k = 0;
        if (b < total) {
            bm_row_of_bit(kColl, b, n, r, k);
            bm_row_setup(kColl, A.spheres_d, A.holes_d, r);
        }
        uint32_t word = 0;
        for (int s = 0; s < 32; ++s) {
            const bool bit = b < total && bm_bit(kColl, r, A.spheres_d, A.holes_d, k);
            const uint64_t m = __ballot(bit);
            if (lane == 2 * s) word = (uint32_t)m;
            if (lane == 2 * s + 1) word = (uint32_t)(m >> 32);
            b += 64;
            k += 64;
            if (b < total && k >= n) {
                do {
                    k -= (int)n;
                    bm_next_row(kColl, n, r);
                } while (k >= n);
                bm_row_setup(kColl, A.spheres_d, A.holes_d, r);
            }
        }
        const int64_t w = run * kWordsPerRun + lane;
        if (w < A.n_words) A.words[w] = word;
    }
}

// Chunk sizes: the tables stay within 2^23 entries each (128 MB of directions,
// 168 MB of rows' terms), or one run of bars and one block of origins.
struct BmPlan {
    int ci, ck;
    int64_t n_dirs, n_rows;
};
BmPlan bitmap_plan(bool coll, int64_t n, int64_t n_org) {
    const int64_t cap = (int64_t)1 << 23;
    const int64_t ci = std::min((n_org + kBmI - 1) / kBmI, std::max<int64_t>(1, cap / kBmI / n)) * kBmI;
    const int64_t o = coll ? ci : n;
    const int64_t ck = std::min((n + 63) / 64, std::max<int64_t>(1, cap / 64 / o)) * 64;
    return BmPlan{(int)ci, (int)ck, o * ck, ci / kBmI * n};
}

}  // namespace

// Without tables where their launches and scratch cost more than 67 instructions a
// bit (calls of both kernels, us): crystal 300 bars (13.5M bits) 51 by the walk,
// 53 by tables, 350 bars (21M) 68 and 61; collimator with 400 holes, 128 bars (6.6M)
// 31 and 33, 192 bars (15M) 43 and 37.
static bool bitmap_by_walk(bool collimator, int64_t n, int64_t n_org) {
    return bm_total_bits(collimator, n, n_org) <= (int64_t)1 << (collimator ? 23 : 24);
}

size_t bitmap_scratch_bytes(bool collimator, int n_det, int n_holes) {
    const int n_org = collimator ? n_holes : n_det;
    if (n_det <= 0 || n_org <= 0 || bitmap_by_walk(collimator, n_det, n_org)) return 0;
    const BmPlan p = bitmap_plan(collimator, n_det, n_org);
    return (size_t)p.n_dirs * sizeof(BmDir) + (size_t)p.n_rows * sizeof(BmRows);
}

hipError_t launch_bitmap(const BitmapLaunch& A, bool collimator, hipStream_t stream) {
    if (A.n_words <= 0) return hipSuccess;
    const int n = A.n_det, n_org = collimator ? A.n_holes : n;
    if (bitmap_by_walk(collimator, n, n_org)) {
        const int64_t n_runs = (A.n_words + kWordsPerRun - 1) / kWordsPerRun;
        const dim3 grid((unsigned)((n_runs + 3) / 4));
        if (collimator)
            hipLaunchKernelGGL(bitmap_walk_kernel<true>, grid, dim3(256), 0, stream, A);
        else
            hipLaunchKernelGGL(bitmap_walk_kernel<false>, grid, dim3(256), 0, stream, A);
        return hipGetLastError();
    }
    const BmPlan p = bitmap_plan(collimator, n, n_org);
    // rows of whole words are stored; others are OR-ed into cleared words (2,000
    // bars: 2.9 ms; 2,048: 2.2 ms)
    const bool whole = n % 32 == 0;
    if (!whole) {
        const int64_t blocks = std::min<int64_t>((A.n_words + 255) / 256, 8192);
        hipLaunchKernelGGL(bitmap_clear_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, A.words, A.n_words);
    }
    BmChunk C;
    C.bars = A.spheres_d;
    C.origins = collimator ? A.holes_d : A.spheres_d;
    C.dirs = (BmDir*)A.scratch;
    C.rows = (BmRows*)((unsigned char*)A.scratch + (size_t)p.n_dirs * sizeof(BmDir));
    C.words = A.words;
    C.n = n;
    for (int k0 = 0; k0 < n; k0 += p.ck) {
        C.k0 = k0;
        C.nk = std::min(p.ck, n - k0);
        C.nk_pad = (C.nk + 63) / 64 * 64;
        for (int i0 = 0; i0 < n_org; i0 += p.ci) {
            C.i0 = i0;
            C.ni = std::min(p.ci, n_org - i0);
            const int64_t blocks_i = (C.ni + kBmI - 1) / kBmI;
            if (collimator || i0 == 0) {  // the crystal's directions serve every chunk of origins
                const int64_t items = (int64_t)(collimator ? C.ni : n) * C.nk_pad;
                const dim3 g((unsigned)((items + 255) / 256));
                if (collimator)
                    hipLaunchKernelGGL(bitmap_dirs_kernel<true>, g, dim3(256), 0, stream, C);
                else
                    hipLaunchKernelGGL(bitmap_dirs_kernel<false>, g, dim3(256), 0, stream, C);
            }
            const int64_t items = blocks_i * kBmI * n;
            hipLaunchKernelGGL(bitmap_rows_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream, C);
            // bars j per wave, whole stores of kBmJ: 32 (2,048 bars: 2.32 ms; 64:
            // 2.36, 128: 2.45, the rows before the diagonal leaving waves idle),
            // down to 16 where the bitmap has few waves
            const int64_t s = blocks_i * (C.nk_pad / 64) * n / 16384 / kBmJ * kBmJ;
            C.slice = (int)std::min<int64_t>(32, std::max<int64_t>(16, s));
            if (collimator)
                launch_chunk<true>(C, whole, stream);
            else
                launch_chunk<false>(C, whole, stream);
        }
    }
    return hipGetLastError();
}

}  // namespace smg
