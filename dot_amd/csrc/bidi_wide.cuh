// Bidirectional softmax for rows of more than 1024 columns: the sweeps of
// bidi_kernels.cuh on strips x chunks tiles.
//
// Workgroup (s, c) of batch element b owns rows [s*rows, (s+1)*rows) and
// columns [c*kCols, (c+1)*kCols).  Row statistics and row dots come out as
// per-chunk partials in a [B, nchunks, L1] plane and are folded in a fixed
// order by one wave per row, in the launch that folds the column statistics or
// dots of the strips ([B, nstrips, L2] partials, as for shorter rows).
// The reference loops a block over any row length (kernels.cu:90-139,
// :153-202); its column kernels walk columns with stride L2.
//
// What bounds it: the sweeps' own 32 bytes per element (sim twice and out, sim
// and grad_out twice and grad); 4 x 3000 x 4096 forward and backward 716 us with
// whole rows per wave, 292 us here (5.4 TB/s of those bytes).  Tiles of 2048
// columns without the loads ahead, as rows beyond 4096 had: 2 x 500 x 9000
// 113 us, 82 here.  Only a row's valid columns are loaded, and a tile without a
// valid column loads nothing.
#pragma once

#include "bidi_kernels.cuh"
#include "tile.cuh"

#pragma clang fp contract(off)

namespace dot_amd {
namespace bidi {
namespace wide_rows {

// Columns of a tile: 16 floats per lane, so that the two row buffers and the
// column state of bwd_dots fit without spilling.
constexpr int kCols = 1024;

inline int num_chunks(int L2) { return (L2 + kCols - 1) / kCols; }

// Pick (VEC, CH) of a tile: float4 columns when rows are 16-byte aligned.
template <class F>
void dispatch(bool vec4, F&& f) {
    using std::integral_constant;
    if (vec4) f(integral_constant<int, 4>{}, integral_constant<int, kCols / (4 * kWave)>{});
    else f(integral_constant<int, 1>{}, integral_constant<int, kCols / kWave>{});
}

struct Tile {
    int s, c;  // strip, chunk
    int c0;    // first column
    int nc;    // columns
    int nv;    // ... of them valid (below the element's l2)
    int nl;    // ... of them loaded: nv rounded up to VEC
};

template <int VEC>
__device__ __forceinline__ Tile tile_of_block(int nchunks, int L2, int l2) {
    Tile t;
    t.c = int(blockIdx.x) % nchunks;
    t.s = int(blockIdx.x) / nchunks;
    t.c0 = t.c * kCols;
    t.nc = min(kCols, L2 - t.c0);
    t.nv = max(0, min(l2 - t.c0, t.nc));
    t.nl = (t.nv + VEC - 1) / VEC * VEC;
    return t;
}

struct Args {
    FwdArgs f;         // forward: statistics planes, strip partials, outputs
    BwdArgs g;         // backward: dots, strip partials, gradient
    float2* rpart;     // [B, nchunks, L1]: row (max, sum) partials (forward)
    float* dpart;      // [B, nchunks, L1]: row dot partials (backward)
    int B, nchunks;
};

// Row statistics partials (base-2 max and sum of 2^(y2 - max) over the chunk)
// and per-strip column states of the chunk's columns.
template <int VEC, int CH>
__global__ __launch_bounds__(kBlock) void fwd_stats(Args w) {
    const int b = batch_of_block();
    if (b >= w.B) return;
    using R = Row<VEC, CH>;
    const FwdArgs& a = w.f;
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int l1, l2;
    valid_extent(a.lengths, b, a.L1, a.L2, l1, l2);
    const Tile tl = tile_of_block<VEC>(w.nchunks, a.L2, l2);
    const bool full = tl.nv == kCols;
    const float sc = a.inv_T * kLog2E;
    const int r0 = tl.s * a.rows;
    const int r1 = min(r0 + a.rows, l1);
    float cm[R::PL], cs[R::PL];
#pragma unroll
    for (int e = 0; e < R::PL; ++e) {
        cm[e] = -FLT_MAX;
        cs[e] = 0.0f;
    }
    float2* part = w.rpart + (size_t(b) * w.nchunks + tl.c) * a.L1;
    const float* base = a.sim + size_t(b) * a.L1 * a.L2 + tl.c0;
    if (tl.nv > 0) {
        auto load = [&](int i, RowBuf<R>& t) { R::load_clamped(base + size_t(i) * a.L2, lane, tl.nl, t.v, 0.0f); };
        pipelined_rows<RowBuf<R>>(r0 + wave, r1, kWavesPerBlock, load, [&](int i, RowBuf<R>& t) {
            float(&y)[R::PL] = t.v;
            float ml = -FLT_MAX;
#pragma unroll
            for (int e = 0; e < R::PL; ++e) {
                y[e] = masked<R>(y[e] * sc, full, lane, e, tl.nv);
                ml = fmaxf(ml, y[e]);
                const float d = y[e] - cm[e];
                const float x = __builtin_amdgcn_exp2f(-fabsf(d));
                const bool gt = d > 0.0f;
                cs[e] = gt ? fmaf(cs[e], x, 1.0f) : cs[e] + x;
                cm[e] = gt ? y[e] : cm[e];
            }
            const float rm = wave_max(ml);
            float sl = 0.0f;
#pragma unroll
            for (int e = 0; e < R::PL; ++e) sl += __builtin_amdgcn_exp2f(y[e] - rm);
            const float rs = wave_sum(sl);
            part[i] = make_float2(rm, rs);  // every lane the same value: no branch
        });
    } else {
        for (int i = r0 + int(threadIdx.x); i < r1; i += kBlock) part[i] = make_float2(-FLT_MAX, 0.0f);
    }
    block_column_combine_lse<VEC, CH>(cm, cs, lds, tl.nc);
    if (wave == 0) {
        const size_t off = (size_t(b) * a.nstrips + tl.s) * a.L2 + tl.c0;
        R::store(a.part_m + off, lane, tl.nc, cm);
        R::store(a.part_s + off, lane, tl.nc, cs);
    }
}

// Workgroups per batch element of the folds: the first cols take kFoldCols
// columns each, the others a row per wave.
struct FoldGrid {
    int cols, rows;
    FoldGrid(int L1, int L2)
        : cols((L2 + kFoldCols - 1) / kFoldCols), rows((L1 + kWavesPerBlock - 1) / kWavesPerBlock) {}
};

// Column statistics from the strips' states, and row statistics of the valid
// rows from the chunk partials (base-2 merge in chunk order).
static __global__ __launch_bounds__(kBlock) void fwd_fold(Args w, int col_blocks) {
    const FwdArgs& a = w.f;
    const int b = batch_of_block();
    if (b >= w.B) return;
    if (int(blockIdx.x) < col_blocks) {
        col_combine_block(a, b);
        return;
    }
    const int i = (int(blockIdx.x) - col_blocks) * kWavesPerBlock + int(threadIdx.x) / kWave;
    int l1, l2;
    valid_extent(a.lengths, b, a.L1, a.L2, l1, l2);
    if (i >= l1) return;
    const int lane = threadIdx.x % kWave;
    const float2* p = w.rpart + size_t(b) * w.nchunks * a.L1 + i;
    float m = -FLT_MAX, s = 0.0f;
    for (int c = lane; c < w.nchunks; c += kWave) {
        const float2 q = p[size_t(c) * a.L1];
        lse_merge2(m, s, q.x, q.y);
    }
    const float M = wave_max(m);
    const float S = wave_sum(s * __builtin_amdgcn_exp2f(m - M));
    if (lane == 0) {
        float* rs = a.row_stats + size_t(b) * 2 * a.L1;
        rs[i] = M;
        rs[a.L1 + i] = S;
    }
}

// r, c, out for one chunk of the strip's rows (as fwd_write); zero rows and
// columns outside the valid region.
template <int VEC, int CH>
__global__ __launch_bounds__(kBlock) void fwd_write(Args w) {
    const int b = batch_of_block();
    if (b >= w.B) return;
    using R = Row<VEC, CH>;
    const FwdArgs& a = w.f;
    // LDS: column max (base 2) kCols | 1 / column sum kCols | row max rows | 1 / row sum rows
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int l1, l2;
    valid_extent(a.lengths, b, a.L1, a.L2, l1, l2);
    const Tile tl = tile_of_block<VEC>(w.nchunks, a.L2, l2);
    const bool full = tl.nv == kCols;
    const float sc = a.inv_T * kLog2E;
    const int r0 = tl.s * a.rows;
    const int r1 = min(r0 + a.rows, a.L1);
    const int rv = tl.nv > 0 ? min(r1, l1) : r0;  // rows with a valid entry in the tile
    float* lcm = lds;
    float* lics = lds + kCols;
    float* lrm = lds + 2 * kCols;
    float* lirs = lrm + a.rows;
    load_col_stats(a.col_stats + size_t(b) * 2 * a.L2 + tl.c0, a.L2, tl.nc, lcm, lics);
    load_row_stats(a.row_stats + size_t(b) * 2 * a.L1, a.L1, r0, rv, lrm, lirs);
    __syncthreads();
    auto write = [&](int i, const float(&o)[R::PL], const float(&rr)[R::PL], const float(&cc)[R::PL]) {
        const size_t off = (size_t(b) * a.L1 + i) * a.L2 + tl.c0;
        R::store_stream(a.out + off, lane, tl.nc, o);
        if (a.row_sm) R::store_stream(a.row_sm + off, lane, tl.nc, rr);
        if (a.col_sm) R::store_stream(a.col_sm + off, lane, tl.nc, cc);
    };
    const float* base = a.sim + size_t(b) * a.L1 * a.L2 + tl.c0;
    auto load = [&](int i, RowBuf<R>& t) { R::load_clamped(base + size_t(i) * a.L2, lane, tl.nl, t.v, 0.0f); };
    pipelined_rows<RowBuf<R>>(r0 + wave, rv, kWavesPerBlock, load, [&](int i, RowBuf<R>& t) {
        const float rm = lrm[i - r0];
        const float irs = lirs[i - r0];
        float o[R::PL], rr[R::PL], cc[R::PL];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            float cm[VEC], ics[VEC];
            R::chunk(lcm, lane, k, tl.nc, cm);
            R::chunk(lics, lane, k, tl.nc, ics);
#pragma unroll
            for (int q = 0; q < VEC; ++q) {
                const int e = k * VEC + q;
                const bool ok = full || R::valid(lane, e, tl.nv);
                const float y2 = t.v[e] * sc;
                rr[e] = ok ? __builtin_amdgcn_exp2f(y2 - rm) * irs : 0.0f;
                cc[e] = ok ? __builtin_amdgcn_exp2f(y2 - cm[q]) * ics[q] : 0.0f;
                o[e] = ok ? __builtin_amdgcn_sqrtf(fmaf(rr[e], cc[e], kEps)) : 0.0f;
            }
        }
        write(i, o, rr, cc);
    });
    float z[R::PL];
#pragma unroll
    for (int e = 0; e < R::PL; ++e) z[e] = 0.0f;
    for (int i = r0 + wave; i < r1; i += kWavesPerBlock)
        if (i >= rv) write(i, z, z, z);
}

// Row dot partials sum_j (d c) r over the chunk and the chunk's column partials
// of (d r) c over the strip.
template <int VEC, int CH, bool RECOMPUTE>
__global__ __launch_bounds__(kBlock) void bwd_dots(Args w) {
    const int b = batch_of_block();
    if (b >= w.B) return;
    using R = Row<VEC, CH>;
    using Src = BwdRow<VEC, CH, RECOMPUTE>;
    const BwdArgs& a = w.g;
    // LDS: statistics 2 nc + 2 rows | block_column_combine's 2 nc
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int l1, l2;
    valid_extent(a.lengths, b, a.L1, a.L2, l1, l2);
    const Tile tl = tile_of_block<VEC>(w.nchunks, a.L2, l2);
    const bool full = tl.nv == kCols;
    const int r0 = tl.s * a.rows;
    const int r1 = min(r0 + a.rows, l1);
    const int rv = tl.nv > 0 ? r1 : r0;
    Src src;
    src.init(a, b, lds, r0, rv, tl.c0, tl.nc, tl.nl);
    __syncthreads();
    float* part = w.dpart + (size_t(b) * w.nchunks + tl.c) * a.L1;
    float acc[R::PL];
#pragma unroll
    for (int e = 0; e < R::PL; ++e) acc[e] = 0.0f;
    bwd_rows<RECOMPUTE>(a, src, b, tl.c0, r0 + wave, rv, lane, [&](int i, const typename Src::Buf& t) {
        float r[R::PL], c[R::PL], d[R::PL];
        src.get(a, i, lane, tl.nv, full, t, r, c, d);
        float dl = 0.0f;
#pragma unroll
        for (int e = 0; e < R::PL; ++e) {
            dl = fmaf(d[e] * c[e], r[e], dl);
            acc[e] = fmaf(d[e] * r[e], c[e], acc[e]);
        }
        part[i] = wave_sum(dl);  // every lane the same value: no branch
    });
    if (tl.nv == 0)
        for (int i = r0 + int(threadIdx.x); i < r1; i += kBlock) part[i] = 0.0f;
    block_column_combine<VEC, CH>(acc, lds + 2 * tl.nc + 2 * a.rows, tl.nc);
    if (wave == 0) R::store(a.partial + (size_t(b) * a.nstrips + tl.s) * a.L2 + tl.c0, lane, tl.nc, acc);
}

// dot_c from the strips' partials, and dot_r of the valid rows from the chunks'.
static __global__ __launch_bounds__(kBlock) void bwd_fold(Args w, int col_blocks) {
    const BwdArgs& a = w.g;
    const int b = batch_of_block();
    if (b >= w.B) return;
    if (int(blockIdx.x) < col_blocks) {
        column_fold_block(a.partial, a.nstrips, b, a.L2, a.dot_c);
        return;
    }
    const int i = (int(blockIdx.x) - col_blocks) * kWavesPerBlock + int(threadIdx.x) / kWave;
    int l1, l2;
    valid_extent(a.lengths, b, a.L1, a.L2, l1, l2);
    if (i >= l1) return;
    const float t = dot_amd::wide::fold_sum(w.dpart + size_t(b) * w.nchunks * a.L1 + i, a.L1, w.nchunks);
    if (threadIdx.x % kWave == 0) a.dot_r[size_t(b) * a.L1 + i] = t;
}

// grad = ((d c - dot_r) r + (d r - dot_c) c) / tau for one chunk, 0 outside
// the valid region, and per-tile sums of grad * sim; tau_partial is [B, gridDim.x].
template <int VEC, int CH, bool RECOMPUTE>
__global__ __launch_bounds__(kBlock) void bwd_write(Args w) {
    const int b = batch_of_block();
    if (b >= w.B) return;
    using R = Row<VEC, CH>;
    using Src = BwdRow<VEC, CH, RECOMPUTE>;
    const BwdArgs& a = w.g;
    __shared__ float scratch[kWavesPerBlock];
    // LDS: statistics 2 nc + 2 rows | column dots nc | row dots rows
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int l1, l2;
    valid_extent(a.lengths, b, a.L1, a.L2, l1, l2);
    const Tile tl = tile_of_block<VEC>(w.nchunks, a.L2, l2);
    const bool full = tl.nv == kCols;
    const int r0 = tl.s * a.rows;
    const int r1 = min(r0 + a.rows, a.L1);
    const int rv = tl.nv > 0 ? min(r1, l1) : r0;
    float* ldc = lds + 2 * tl.nc + 2 * a.rows;
    float* ldr = ldc + tl.nc;
    for (int j = threadIdx.x; j < tl.nc; j += kBlock) ldc[j] = a.dot_c[size_t(b) * a.L2 + tl.c0 + j];
    for (int t = threadIdx.x; t < rv - r0; t += kBlock) ldr[t] = a.dot_r[size_t(b) * a.L1 + r0 + t];
    Src src;
    src.init(a, b, lds, r0, rv, tl.c0, tl.nc, tl.nl);
    __syncthreads();
    float tacc = 0.0f;
    const bool want_tau = a.tau_partial != nullptr;
    auto store = [&](int i, const float(&gs)[R::PL]) {
        R::store_stream(a.grad_sim + (size_t(b) * a.L1 + i) * a.L2 + tl.c0, lane, tl.nc, gs);
    };
    bwd_rows<RECOMPUTE>(a, src, b, tl.c0, r0 + wave, rv, lane, [&](int i, const typename Src::Buf& t) {
        float r[R::PL], c[R::PL], d[R::PL], gs[R::PL];
        src.get(a, i, lane, tl.nv, full, t, r, c, d);
        const float dr = ldr[i - r0];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            float dc[VEC];
            R::chunk(ldc, lane, k, tl.nc, dc);
#pragma unroll
            for (int q = 0; q < VEC; ++q) {
                const int e = k * VEC + q;
                const bool valid = full || R::valid(lane, e, tl.nv);
                const float tt = (d[e] * c[e] - dr) * r[e] + (d[e] * r[e] - dc[q]) * c[e];
                gs[e] = valid ? tt * a.inv_T : 0.0f;
                if (want_tau) tacc = valid ? fmaf(gs[e], t.y[e], tacc) : tacc;
            }
        }
        store(i, gs);
    });
    float z[R::PL];
#pragma unroll
    for (int e = 0; e < R::PL; ++e) z[e] = 0.0f;
    for (int i = r0 + wave; i < r1; i += kWavesPerBlock)
        if (i >= rv) store(i, z);
    if (want_tau) {
        const float tsum = block_reduce<kWavesPerBlock>(wave_sum(tacc), scratch, OpSum{});
        if (threadIdx.x == 0) a.tau_partial[size_t(b) * gridDim.x + blockIdx.x] = tsum;
    }
}

}  // namespace wide_rows
}  // namespace bidi
}  // namespace dot_amd
