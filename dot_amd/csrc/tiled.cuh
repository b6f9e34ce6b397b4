// Tiled persistent forward: one launch for all iterations, each batch element
// cut in two dimensions over W = C x ST workgroups.
//
// Workgroup (s, c) of element b owns the tile of rows [s R, (s+1) R) and
// columns [c seg, (c+1) seg).  The iteration runs in the scaling domain of
// res::forward: E_ij = 2^(K_ij log2(e) - max_j) once (res::ScaledKernel), then
//   w_i = a_i / sum_j E_ij V_j,   V_j = b_j / sum_i E_ij w_i,   P = E w V,
// two FMAs per element and iteration.  Each wave takes every eighth row of
// the tile in batches of KB rows and completes a batch's row sums by itself:
// it publishes its tile's partial of each row as a tagged word (resident.cuh)
// and polls the C words of the row's tiles, while other waves' loads are in
// flight.  The column sums are folded over the workgroup's waves, published,
// summed by the owner of a slice of the tile's columns (strip s owns 1/ST of
// them) and gathered, as in persistent.cuh, but over the tile's columns only.
//
// Why tiles: a workgroup that owns whole rows exchanges N words three times per
// iteration whatever its share of the rows is (4 x 4096 x 4096: 14 of 40 us per
// iteration; rows of 16384 columns would exchange more than they stream), and
// its column accumulator takes 64 floats per lane.  A tile of 512 columns
// exchanges 512 words, and its 8-float accumulator leaves registers for two
// batches and for RR rows per wave of E that stay in them; the rest is streamed
// from E, which is kept in the plan's buffer until the plan replaces it.
// Measured per iteration, row tier (log domain) or sweeps -> tiles: 16 x 1024 x
// 2048 22.5 -> 18.4 us, 4 x 4096 x 4096 39.7 -> 39.3, 144 x 400 x 450 42 -> 21,
// 77 x 768 x 568 37 -> 21, 4 x 1024 x 16384 101 -> 39.  What bounds it: a wave's batches, each a load
// (2-3 us behind eight waves' streams) with its row exchange; neither rows of E
// kept in LDS as well nor a third buffer made a difference.
//
// An element leaves the scaling domain for the log domain for good when a
// factor or a column sum passes its bounds (res::kScaleMax ...): the owner of
// such a column forms the exact column log-sum-exp and publishes v itself
// under a tag with kLogBit set, the workgroups that gather it tag their row
// words of the next iteration with it, and so every workgroup of the element redoes
// that iteration's rows in the log domain, from the scores.
//
// The stop test sees |u_t - u_{t-1}| as ln(w_t / w_{t-1}), resolved to the
// rounding of a row's sum (~2e-7) whatever the size of the potentials, so it
// fires where 64-bit arithmetic has it fire (25 x 670 x 1651 at reg 0.987:
// iteration 3; the rounded potentials wobble by more than tol = 1e-6 and ran
// all 262).
#pragma once

#include <cfloat>
#include <cstdint>

#include "persistent.cuh"

namespace dot_amd {
namespace til {

using res::kThreads;
using res::kWaves;
using res::publish;
using res::tag_pack;
typedef unsigned long long word_t;

constexpr int kMaxTiles = 16;                 // column tiles per batch element (C)
constexpr int kMaxStrips = 256;               // row strips per batch element (ST)
constexpr unsigned kLogBit = 0x80000000u;     // tag bit: a column's word is v, not V; a row's tile leaves
constexpr unsigned kSetupTag = 0x7ffffffeu;   // rows' largest scores (an iteration tag is below it)
constexpr int kColsPerThread = 3;             // ceil((1024 + kMaxStrips) / kThreads)

struct FwdArgs {
    const float* X;       // scores [B,M,N]
    float kscale;         // K = X * kscale
    int scores_kind;      // +1 log_alpha, -1 cost
    const float* log_a;   // [B,M] or null
    const float* log_b;   // [B,N] or null
    float log_a_default, log_b_default;
    float tol;
    int max_iter;
    float* plan;          // [B,M,N]: E during the iterations, then the plan
    float* cost_partial;  // [G] by logical workgroup, or null
    float* u_out;         // [B,M] or null
    float* v_out;         // [B,N] or null
    float* u_hist;        // [T,B,M] or null
    float* v_hist;        // [T,B,N] or null
    int32_t* iters_used;
    int32_t* converged;
    word_t* rowx;         // [2,B,M,C] row partials
    word_t* rowl;         // [2,B,M,C,2] log domain: (maximum, sum) of a row's tile
    word_t* part;         // [2,G,seg] workgroup column sums
    word_t* res;          // [2,B,N] new V (or v)
    word_t* uslot;        // [2,B,M] u (read by the exact column LSE)
    word_t* dxchg;        // [kDeltaSlots,G] per-workgroup deltas
    word_t* xcc;          // [G] XCC ids
    int* status;
    int B, M, N, C, ST, R, seg, spin_limit;
    int G;                // B ST C: workgroups with a tile (the grid may be padded, see forward)
    int local_ok;         // XCD-local exchange stores allowed (local_exchange_allowed)
};

// LDS floats of the forward.
inline __host__ __device__ size_t fwd_lds_floats(int seg, int ST, int R) {
    // fold 8 seg | V 2 seg | log b seg | red seg + ST | rows 4R | u 2R | log a R | scratch 32
    const size_t red = (size_t(seg) + ST + 3) & ~size_t(3);
    return ((size_t(kWaves) + 3) * seg + red + 7 * size_t(R) + 32 + 3) & ~size_t(3);
}

// Polls one tagged word per lane (lanes with `on`) until all carry tag t (or t |
// kLogBit: `left`, for the wave); NaN after a timeout.  `dead` is kept uniform
// over the wave.
__device__ __forceinline__ float poll_lane(const word_t* p, bool on, unsigned t, int spin_limit, int* status,
                                           bool& dead, bool& left) {
    res::forced_timeout(spin_limit, status, dead);
    for (int spins = 0; !dead; ++spins) {
        word_t x = tag_pack(0.0f, t);
        if (on) x = __hip_atomic_load(const_cast<word_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned tag = static_cast<unsigned>(x >> 32);
        if (__all((tag & ~kLogBit) == t)) {
            left = __any(tag != t);
            return __uint_as_float(static_cast<unsigned>(x));
        }
        const bool failed =
            (spins & 255) == 255 && __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        if (spins >= spin_limit) atomicOr(status, 1);
        dead = __any(failed) || spins >= spin_limit;
    }
    return __builtin_nanf("");
}

// Polls the words at idx(r), r < n <= kColsPerThread, until each carries tag t
// (or t | kLogBit, noted in `logs`); NaN after a timeout.
template <class Idx>
__device__ __forceinline__ void poll_cols(const word_t* base, int n, Idx idx, unsigned t, int spin_limit,
                                          int* status, bool& dead, float (&out)[kColsPerThread],
                                          unsigned& logs) {
    res::forced_timeout(spin_limit, status, dead);
    for (int spins = 0; !dead; ++spins) {
        bool ready = true;
        unsigned lg = 0;
#pragma unroll
        for (int r = 0; r < kColsPerThread; ++r) {
            if (r < n) {
                const word_t x = __hip_atomic_load(const_cast<word_t*>(base + idx(r)), __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
                const unsigned tag = static_cast<unsigned>(x >> 32);
                ready = ready && (tag & ~kLogBit) == t;
                lg |= (tag >> 31) << r;
                out[r] = __uint_as_float(static_cast<unsigned>(x));
            }
        }
        if (ready) {
            logs = lg;
            return;
        }
        if (((spins & 255) == 255 &&
             __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) ||
            spins >= spin_limit) {
            if (spins >= spin_limit) atomicOr(status, 1);
            dead = true;
        }
    }
    logs = 0;
#pragma unroll
    for (int r = 0; r < kColsPerThread; ++r) out[r] = __builtin_nanf("");
}

// Reduction over groups of 2^lg consecutive lanes (lg <= 4); every lane of a
// group gets the same bits.
template <class Op>
__device__ __forceinline__ float group_reduce(float x, int lg, Op op) {
    if (lg >= 1) x = op(x, dpp_move<kDppQuadXor1>(x));
    if (lg >= 2) x = op(x, dpp_move<kDppQuadXor2>(x));
    if (lg >= 3) x = op(x, dpp_move<kDppRowHalfMirror>(x));
    if (lg >= 4) x = op(x, dpp_move<kDppRowMirror>(x));
    return x;
}

// A wave's batch of KB rows across the element's tiles: rows k0, k0 + 1, ... <
// kend of the wave (row k is row wave + 8 k of the tile).  `own` is a
// transposed reduction's result (row r at lane_of_slot<KB>(r)); the finished
// value of batch row r is in the lanes of group r (lanes r 2^lg ... of 2^lg
// each).  A row's C words are adjacent; offsets are bytes from the slots, below
// 4 GiB (tiled_config).
template <int KB>
struct RowGroup {
    static constexpr int kStep = 16 / KB;  // lanes per row of a transposed reduction
    int lane, wave, lg, C;
    unsigned put_at, get_at, step;  // this lane's word of row 0, of its group's row 0; bytes per k

    __device__ __forceinline__ RowGroup(int lane_, int wave_, int C_, int c, size_t row_base) {
        lane = lane_;
        wave = wave_;
        C = C_;
        lg = 0;
        while ((1 << lg) < C) ++lg;
        const unsigned first = unsigned(row_base) + unsigned(wave);
        put_at = ((first + kWaves * unsigned(lane / kStep)) * unsigned(C) + unsigned(c)) * unsigned(sizeof(word_t));
        get_at = ((first + kWaves * unsigned(group())) * unsigned(C) + unsigned(lane & ((1 << lg) - 1))) *
                 unsigned(sizeof(word_t));
        step = unsigned(kWaves) * unsigned(C) * unsigned(sizeof(word_t));
    }
    __device__ __forceinline__ int group() const { return lane >> lg; }
    __device__ __forceinline__ int group_row(int k0) const { return wave + kWaves * (k0 + group()); }
    __device__ __forceinline__ bool group_ok(int k0, int kend) const { return group() < KB && k0 + group() < kend; }
    __device__ __forceinline__ bool leader() const { return (lane & ((1 << lg) - 1)) == 0; }
    __device__ __forceinline__ float of_group(float x, int r) const { return read_lane(x, r << lg); }

    // `words` per row and tile, this value at `which`
    __device__ __forceinline__ void put(word_t* slots, float own, int k0, int kend, unsigned t, bool local,
                                        int words = 1, int which = 0) const {
        if (lane < 16 && lane % kStep == 0 && k0 + lane / kStep < kend)
            publish(reinterpret_cast<word_t*>(reinterpret_cast<char*>(slots) +
                                              (put_at + unsigned(k0) * step) * unsigned(words)) + which,
                    own, t, local);
    }
    __device__ __forceinline__ bool reads(int k0, int kend) const {
        return group_ok(k0, kend) && (lane & ((1 << lg) - 1)) < C;
    }
    __device__ __forceinline__ float get(const word_t* slots, int k0, int kend, unsigned t, int spin_limit,
                                         int* status, bool& dead, bool& left, int words = 1, int which = 0) const {
        return poll_lane(reinterpret_cast<const word_t*>(reinterpret_cast<const char*>(slots) +
                                                         (get_at + unsigned(k0) * step) * unsigned(words)) + which,
                         reads(k0, kend), t, spin_limit, status, dead, left);
    }
    __device__ __forceinline__ float get(const word_t* slots, int k0, int kend, unsigned t, int spin_limit,
                                         int* status, bool& dead, int words = 1, int which = 0) const {
        bool left;  // (nobody leaves here)
        return get(slots, k0, kend, t, spin_limit, status, dead, left, words, which);
    }
    // one tile per row: the value moves to its group's lane without memory
    __device__ __forceinline__ float to_group(float own) const {
        float x = 0.0f;
#pragma unroll
        for (int r = 0; r < KB; ++r) {
            const float q = read_lane(own, res::lane_of_slot<KB>(r));
            if (lane == r) x = q;
        }
        return x;
    }
};

// Exact max-shifted log-sum-exp of K + u_t (kernels.cu:629-671) over columns of
// one element: the lanes set in `need` get that of column col0 + lane.  bM is
// the element's first row; the potentials are awaited under tag t.  The wave's
// lanes are dealt to the columns (all 64 to one, one to each of 64), each taking
// four rows at a time, so that a wait covers 4 x 64 rows where a thread per
// column waited for each row's word.  One far column, 20 iterations at reg 0.01:
// 3 x 2272 x 80 1316 -> 244 us per call, 4 x 1024 x 16384 2132 -> 1362 (1110
// without the far column; with the log domain's rows loaded a batch ahead).
__device__ __forceinline__ float exact_columns(const FwdArgs& a, unsigned long long need, unsigned t, size_t bM,
                                            int col0, bool& dead) {
    const int lane = threadIdx.x % kWave;
    int lg = 6;  // 2^lg lanes per column
    while ((__popcll(need) << lg) > kWave) --lg;
    const int sub = lane & ((1 << lg) - 1);
    unsigned long long left = need;
    for (int k = lane >> lg; k > 0; --k) left &= left - 1;
    const bool on = left != 0;
    const float* col = a.X + bM * a.N + col0 + (on ? __ffsll(left) - 1 : 0);
    const word_t* urow = a.uslot + size_t(t & 1) * a.B * a.M + bM;
    constexpr int Q = 4;
    const int step = 1 << lg;
    auto terms = [&](int i0, float(&y)[Q]) {  // K + u of this lane's next rows, -inf past the last
        word_t u[Q];
        float x[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int i = min(i0 + q * step, a.M - 1);
            u[q] = __hip_atomic_load(const_cast<word_t*>(urow + i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            x[q] = col[size_t(i) * a.N];
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int i = i0 + q * step;
            float ui = __uint_as_float(static_cast<unsigned>(u[q]));
            if (i < a.M && static_cast<unsigned>(u[q] >> 32) != t)
                ui = res::collect(const_cast<word_t*>(urow + i), t, a.spin_limit, a.status, dead);
            y[q] = i < a.M ? x[q] * a.kscale + ui : -INFINITY;
        }
    };
    float mx = -FLT_MAX, sm = 0.0f;
    if (on)
        for (int i = sub; i < a.M; i += Q * step) {
            float y[Q];
            terms(i, y);
#pragma unroll
            for (int q = 0; q < Q; ++q) mx = fmaxf(mx, y[q]);
        }
    for (int d = step / 2; d > 0; d /= 2) mx = fmaxf(mx, __shfl_xor(mx, d));
    if (on)
        for (int i = sub; i < a.M; i += Q * step) {
            float y[Q];
            terms(i, y);
#pragma unroll
            for (int q = 0; q < Q; ++q) sm += safe_exp(y[q] - mx);
        }
    for (int d = step / 2; d > 0; d /= 2) sm += __shfl_xor(sm, d);
    const float lse = mx + logf(fmaxf(sm, sk::kSumFloor));
    return __shfl(lse, __popcll(need & ((1ull << lane) - 1)) << lg);
}

template <int VEC, int CH, int KB, int RR>
__global__ __launch_bounds__(kThreads) void forward(FwdArgs a) {
    using Rw = Row<VEC, CH>;
    constexpr int PL = Rw::PL;
    static_assert(RR % KB == 0 && KB >= 1 && KB <= 8, "whole batches of resident rows");
    extern __shared__ float lds[];
    const int seg = a.seg, R = a.R, C = a.C, ST = a.ST;
    float* fold = lds;
    float* lds_v = fold + kWaves * seg;  // [2][seg] V by iteration parity (v in the log domain)
    float* lds_lb = lds_v + 2 * seg;
    float* red = lds_lb + seg;
    // a row of the scaling domain: a, the row's largest score (times the sign of K), sum E V by iteration parity
    float4* lds_row4 = reinterpret_cast<float4*>(lds + ((size_t(kWaves) + 3) * seg + ((seg + ST + 3) & ~3)));
    float* lds_u = reinterpret_cast<float*>(lds_row4 + R);  // log domain: u by iteration parity
    float* lds_la = lds_u + 2 * R;
    float* scratch = lds_la + R;  // [0] global delta, [1..kWaves] wave deltas, [16..] reductions
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // The dispatcher deals workgroups to the 8 XCDs in turn.  Consecutive strips go
    // to one XCD, a strip's C tiles always, so that their words stay in its L2; the
    // grid has room for as many strips on each (a strip that is not there returns).
    const int G = a.G;
    const int turn = int(blockIdx.x) / res::kXcds;
    const int strip = int(blockIdx.x) % res::kXcds * (int(gridDim.x) / res::kXcds / C) + turn / C;
    if (strip >= a.B * ST) return;
    const int c = turn % C, s = strip % ST, b = strip / ST;
    const int gid = strip * C + c;
    const int row0 = s * R;
    const int nrows = min(R, a.M - row0);
    const int c0 = c * seg;
    const int nc = min(seg, a.N - c0);
    const int j0 = pst::slice_begin(s, ST, nc), j1 = pst::slice_begin(s + 1, ST, nc);
    const size_t bM = size_t(b) * a.M, bN = size_t(b) * a.N;
    const size_t tile0 = (bM + row0) * a.N + c0;
    const int nk = nrows > wave ? (nrows - wave + kWaves - 1) / kWaves : 0;  // this wave's rows
    const bool check = a.tol > 0.0f;
    const float pad = a.kscale > 0.0f ? -INFINITY : INFINITY;  // a score whose K is -inf
    const float kscale2 = a.kscale * kLog2E;
    const RowGroup<KB> rg(lane, wave, C, c, bM + row0);
    bool dead = false;
    if (threadIdx.x == 0)
        publish(a.xcc + gid, __int_as_float(res::xcc_id()), res::kXccTag);

    for (int l = threadIdx.x; l < R; l += kThreads) {
        const float la = (l < nrows && a.log_a) ? a.log_a[bM + row0 + l] : a.log_a_default;
        lds_la[l] = la;
        lds_row4[l] = make_float4(safe_exp(la), 0.0f, 0.0f, 0.0f);
    }
    for (int j = threadIdx.x; j < nc; j += kThreads) {
        lds_lb[j] = a.log_b ? a.log_b[bN + c0 + j] : a.log_b_default;
        lds_v[j] = lds_v[seg + j] = 1.0f;
    }
    __syncthreads();

    // Rows through buffer resources of their tile's columns: one lane offset for
    // all of a row's loads, and columns past the tile read 0.  A batch's rows are
    // clamped to this wave's last one (a cache hit), so that every load is
    // unconditional.
    const size_t row_step = size_t(kWaves) * a.N;
    auto load_row = [&](const float* row, float(&x)[PL]) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, nc * int(sizeof(float)), 0x00020000);
        const unsigned at = unsigned(lane) * VEC * unsigned(sizeof(float));
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            if constexpr (VEC == 4) {
                typedef unsigned v4u __attribute__((ext_vector_type(4)));
                const v4u q = __builtin_amdgcn_raw_buffer_load_b128(rs, at, k * 1024, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * k + e] = __uint_as_float(q[e]);
            } else {
                x[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, at, k * 256, 0));
            }
        }
    };
    auto load_rows = [&](const float* base, int k0, float(&x)[KB][PL]) {
        const float* first = base + tile0 + size_t(wave) * a.N;
#pragma unroll
        for (int r = 0; r < KB; ++r) load_row(first + size_t(min(k0 + r, nk - 1)) * row_step, x[r]);
    };
    auto mask_rows = [&](float(&x)[KB][PL]) {  // scores: the value whose K is -inf past the tile
#pragma unroll
        for (int r = 0; r < KB; ++r)
#pragma unroll
            for (int e = 0; e < PL; ++e)
                if (!Rw::valid(lane, e, nc)) x[r][e] = pad;
    };

    // E of a batch, from the rows' largest scores over the tiles
    const res::ScaledKernel kernel(a.kscale);
    auto form_e = [&](float(&x)[KB][PL], int k0) {
        mask_rows(x);
        float lm[KB];
#pragma unroll
        for (int r = 0; r < KB; ++r) {
            lm[r] = -INFINITY;
#pragma unroll
            for (int e = 0; e < PL; ++e) lm[r] = fmaxf(lm[r], x[r][e] * kernel.sign);
        }
        const float own = res::transposed_reduce<KB>(lm, OpMax{});
        float top;
        if (C > 1) {
            rg.put(a.rowx, own, k0, nk, kSetupTag, false);
            top = rg.get(a.rowx, k0, nk, kSetupTag, a.spin_limit, a.status, dead);
            top = group_reduce(rg.reads(k0, nk) ? top : -INFINITY, rg.lg, OpMax{});
        } else {
            top = rg.to_group(own);
        }
        if (rg.leader() && rg.group_ok(k0, nk)) lds_row4[rg.group_row(k0)].y = top;
#pragma unroll
        for (int r = 0; r < KB; ++r) {
            const auto row = kernel.row(rg.of_group(top, r));
            const bool in = k0 + r < nk;  // rows past the last: 0
#pragma unroll
            for (int e = 0; e < PL; ++e) x[r][e] = in ? kernel.e(x[r][e], row) : 0.0f;
        }
    };

    float xr[RR > 0 ? RR / KB : 1][KB][PL];  // rows k < RR of this wave, by batch
    if (nk > 0) {
#pragma unroll
        for (int q = 0; q < RR / KB; ++q) load_rows(a.X, q * KB, xr[q]);
#pragma unroll
        for (int q = 0; q < RR / KB; ++q) form_e(xr[q], q * KB);
        // the others' E to the plan's buffer (forming it in the first iteration's row
        // pass instead spilled the resident rows: +2 us per iteration)
        float x[KB][PL], y[KB][PL];
        auto setup = [&](float(&q)[KB][PL], int k0, float(&next)[KB][PL]) {
            load_rows(a.X, k0 + KB, next);
            form_e(q, k0);
#pragma unroll
            for (int r = 0; r < KB; ++r)
                if (k0 + r < nk) Rw::store(a.plan + tile0 + size_t(wave + kWaves * (k0 + r)) * a.N, lane, nc, q[r]);
        };
        load_rows(a.X, RR, x);
        for (int k = RR; k < nk; k += 2 * KB) {
            setup(x, k, y);
            if (k + KB < nk) setup(y, k + KB, x);
        }
    } else {  // a wave without rows adds 0 w = 0 to the column sums: its registers must not hold infinities or NaN
#pragma unroll
        for (int q = 0; q < RR / KB; ++q)
#pragma unroll
            for (int r = 0; r < KB; ++r)
#pragma unroll
                for (int e = 0; e < PL; ++e) xr[q][r][e] = 0.0f;
    }

    // XCD checks: the words of a row stay in its strip, those of a column in its tiles
    bool local_row, local_col;
    {
        const int me = res::xcc_id();
        bool same_row = true, same_col = true;
        if (wave == 0) {
            for (int q = lane; q < C; q += kWave)
                same_row = same_row && __float_as_int(res::collect(a.xcc + (size_t(b) * ST + s) * C + q, res::kXccTag,
                                                                   a.spin_limit, a.status, dead)) == me;
            for (int q = lane; q < ST; q += kWave)
                same_col = same_col && __float_as_int(res::collect(a.xcc + (size_t(b) * ST + q) * C + c, res::kXccTag,
                                                                   a.spin_limit, a.status, dead)) == me;
            dead = __any(dead);
        }
        local_row = !__syncthreads_or(!same_row) && a.local_ok;
        local_col = !__syncthreads_or(!same_col) && a.local_ok;
    }

    bool scal = true;    // scaling domain
    bool leave = false;  // ... until the next iteration's row update
    int used = a.max_iter;
    int conv = 0;
    float acc[PL], dmax = 0.0f;
    auto clear = [&]() {
        dmax = 0.0f;
#pragma unroll
        for (int e = 0; e < PL; ++e) acc[e] = 0.0f;
    };
    // wave 0: the loads of iteration t - 1's deltas, and their maximum into scratch[0]
    auto prefetch_deltas = [&](int t, word_t(&dpre)[res::kDeltaPrefetch]) {
        const word_t* ds = a.dxchg + size_t((t - 1) % res::kDeltaSlots) * G;
#pragma unroll
        for (int q = 0; q < res::kDeltaPrefetch; ++q) {
            const int g = lane + q * kWave;
            dpre[q] = g < G ? __hip_atomic_load(const_cast<word_t*>(ds + g), __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT)
                            : tag_pack(0.0f, unsigned(t - 1));
        }
    };
    auto finish_deltas = [&](int t, const word_t(&dpre)[res::kDeltaPrefetch]) {
        word_t* ds = a.dxchg + size_t((t - 1) % res::kDeltaSlots) * G;
        float gmax = 0.0f;
#pragma unroll
        for (int q = 0; q < res::kDeltaPrefetch; ++q) {
            const int g = lane + q * kWave;
            if (g < G) {
                float d = __uint_as_float(static_cast<unsigned>(dpre[q]));
                if (static_cast<unsigned>(dpre[q] >> 32) != unsigned(t - 1))
                    d = res::collect(ds + g, unsigned(t - 1), a.spin_limit, a.status, dead);
                gmax = res::OpMaxNan{}(gmax, d);
            }
        }
        for (int g = lane + res::kDeltaPrefetch * kWave; g < G; g += kWave)
            gmax = res::OpMaxNan{}(gmax, res::collect(ds + g, unsigned(t - 1), a.spin_limit, a.status, dead));
        gmax = wave_reduce(gmax, res::OpMaxNan{});
        if (lane == 0) scratch[0] = gmax;
    };
    // u of a row: to the exact column log-sum-exp's readers and the history
    auto put_u = [&](int t, float u, int l) {
        publish(a.uslot + size_t(t & 1) * a.B * a.M + bM + row0 + l, u, unsigned(t));
        if (a.u_hist) a.u_hist[(size_t(t - 1) * a.B + b) * a.M + row0 + l] = u;
    };
    // u of a row from its sum of E V (a zero marginal's is -inf)
    auto u_of = [&](float log_a, float top, float sum) {
        return log_a - kLn2 * kernel.log2_sum(kernel.row(top), __builtin_amdgcn_logf(sum));
    };
    // the potentials of iteration t from its row sums, for the log domain
    auto rows_to_u = [&](int t) {
        for (int l = threadIdx.x; l < nrows; l += kThreads) {
            const float4 q = lds_row4[l];
            lds_u[(t & 1) * R + l] = t > 0 ? u_of(lds_la[l], q.y, (t & 1) ? q.w : q.z) : 0.0f;
        }
    };
    // The column sums of iteration t, exchanged into the tile's new factors:
    // V in lds_v (v in the log domain).  Returns this thread's columns whose word
    // is v (a bit each).
    auto columns = [&](auto scaling_domain, int t) -> unsigned {
        constexpr bool SC = decltype(scaling_domain)::value;
        const int cur = t & 1, prev = cur ^ 1;
        const unsigned tag = unsigned(t);
        dmax = wave_max(dmax);
        if (lane == 0) scratch[1 + wave] = dmax;
        pst::publish_row_flat<VEC, CH>(acc, fold, nc, a.part + (size_t(cur) * G + gid) * seg, tag, local_col);
        if (check) {
            float d = scratch[1];
#pragma unroll
            for (int q = 1; q < kWaves; ++q) d = fmaxf(d, scratch[1 + q]);
            if (threadIdx.x == 0) publish(a.dxchg + size_t(t % res::kDeltaSlots) * G + gid, d, tag);
        }

        // The owner's totals of its columns [j0, j1) of the tile, over the ST strips in order.
        word_t* res_row = a.res + size_t(cur) * a.B * a.N + bN + c0;
        {
            int tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            const int S = j1 - j0, n = ST * S;
            const int mine = n > tid ? (n - 1 - tid) / kThreads + 1 : 0;
            float got[kColsPerThread];
            unsigned logs;
            poll_cols(a.part + (size_t(cur) * G + size_t(b) * ST * C + c) * seg, mine,
                      [&](int r) {
                          const int q = tid + r * kThreads;  // q = strip * S + jj
                          return size_t(q / S) * C * seg + j0 + q % S;
                      },
                      tag, a.spin_limit, a.status, dead, got, logs);
#pragma unroll
            for (int r = 0; r < kColsPerThread; ++r)
                if (r < mine) red[tid + r * kThreads] = got[r];
            __syncthreads();
            for (int first = 0; first < S; first += kThreads) {
                const int jj = first + int(threadIdx.x);
                const bool in = jj < S;
                float cs = 0.0f;
                if (in)
                    for (int g = 0; g < ST; ++g) cs += red[g * S + jj];
                if (dead) cs = __builtin_nanf("");
                const int j = j0 + jj;
                const float lb = in ? lds_lb[j] : 0.0f;
                float vn = 0.0f;
                bool lin = SC, good;
                if constexpr (SC) {
                    vn = safe_exp(lb) / cs;
                    good = cs >= res::scaled_col_min(a.M) && vn >= res::kScaleMin && vn <= res::kScaleMax;
                } else {
                    good = cs >= sk::kColSumFloor && cs <= FLT_MAX;
                    if (in && good) vn = lb + lds_v[prev * seg + j] - logf(cs);
                }
                if (!good) {
                    vn = -INFINITY;  // a zero marginal's v, whatever the column (in every iteration: no sum to form)
                    lin = false;
                }
                const unsigned long long need = __ballot(in && !good && lb != -INFINITY);
                // (kept out of the loop's line: in it, 144 x 400 x 450 took 20.3 us per iteration for 18.9)
                if (__builtin_expect(need != 0, 0)) {
                    const float x = exact_columns(a, need, tag, bM, c0 + j - lane, dead);
                    if ((need >> lane) & 1u) vn = lb - x;
                }
                if (in) {
                    publish(res_row + j, vn, (SC && !lin) ? (tag | kLogBit) : tag, local_col);
                    if (a.v_hist) a.v_hist[(size_t(t - 1) * a.B + b) * a.N + c0 + j] = lin ? logf(vn) : vn;
                }
            }
        }
        // All of the tile's new factors.
        unsigned logs = 0;
        {
            int tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            const int ncol = nc > tid ? (nc - 1 - tid) / kThreads + 1 : 0;
            float got[kColsPerThread];
            poll_cols(res_row, ncol, [&](int r) { return size_t(tid + r * kThreads); }, tag, a.spin_limit,
                      a.status, dead, got, logs);
#pragma unroll
            for (int r = 0; r < kColsPerThread; ++r)
                if (r < ncol) lds_v[cur * seg + tid + r * kThreads] = got[r];
        }
        return logs;
    };

    int t0 = 1;  // the log domain's first iteration
    for (int t = 1; scal && t <= a.max_iter; ++t) {
        const int cur = t & 1, prev = cur ^ 1;
        const unsigned tag = unsigned(t);
        const bool test = check && t >= 2;
        word_t* rowx = a.rowx + size_t(cur) * a.B * a.M * C;
        bool left = leave, bad = false;
        clear();
        if (leave) {
            // (a row of one tile has no row words: everyone who would read them leaves as well)
            for (int l = threadIdx.x; C > 1 && l < nrows; l += kThreads)
                publish(rowx + (bM + row0 + l) * C + c, 0.0f, tag | kLogBit);
        } else {
            float v[PL];
            Rw::load(lds_v + prev * seg, lane, nc, v, 0.0f);
            auto dots = [&](const float(&x)[KB][PL]) {
                float d[KB];
#pragma unroll
                for (int r = 0; r < KB; ++r) {
                    d[r] = 0.0f;
#pragma unroll
                    for (int e = 0; e < PL; ++e) d[r] = fmaf(x[r][e], v[e], d[r]);
                }
                return res::transposed_sum<KB>(d);
            };
            // w and u of a batch, and its rows' share of the column sums
            auto finish = [&](const float(&x)[KB][PL], int k0, float own) {
                float s_sum;
                if (C > 1) {
                    const bool on = rg.reads(k0, nk);
                    bool peer_left = false;
                    s_sum = rg.get(rowx, k0, nk, tag, a.spin_limit, a.status, dead, peer_left);
                    if (peer_left) {  // all of the strip's rows say so
                        left = true;
                        return;
                    }
                    s_sum = group_reduce(on ? s_sum : 0.0f, rg.lg, OpSum{});
                } else {
                    s_sum = rg.to_group(own);
                }
                const bool ok = rg.group_ok(k0, nk);
                const int l = ok ? rg.group_row(k0) : 0;
                const float4 rw = lds_row4[l];
                const float lga = lds_la[l];
                const float s_l = s_sum > 0.0f ? s_sum : sk::kSumFloor;  // 0: a row with no finite K
                const float w = ok ? rw.x / s_l : 0.0f;
                bad = bad || (ok && !(s_sum == 0.0f || (s_sum > 0.0f && w <= res::kScaleMax)));
                if (check) {
                    // |u_t - u_{t-1}| = |ln(s_t / s_{t-1})|, by its series once the sums agree
                    // to 1 %: resolved to their rounding (~2e-7).  A row of a zero marginal,
                    // whose u is -inf, does not change after the first iteration.
                    const float s_prev = cur ? rw.z : rw.w;
                    const float q = (s_prev - s_l) * __builtin_amdgcn_rcpf(s_l);
                    float d = ok ? fabsf(q - 0.5f * q * q) : 0.0f;
                    if (__any(ok && !(fabsf(q) <= 0.01f))) {
                        if (ok && !(fabsf(q) <= 0.01f))
                            d = fabsf(t > 1 ? kLn2 * __builtin_amdgcn_logf(s_prev / s_l) : u_of(lga, rw.y, s_l));
                    }
                    if (t > 1 && lga == -INFINITY) d = 0.0f;
                    dmax = fmaxf(dmax, d);
                }
                if (ok && rg.leader()) (cur ? lds_row4[l].w : lds_row4[l].z) = s_l;
#pragma unroll
                for (int r = 0; r < KB; ++r) {
                    const float wr = rg.of_group(w, r);
#pragma unroll
                    for (int e = 0; e < PL; ++e) acc[e] = fmaf(x[r][e], wr, acc[e]);
                }
#pragma unroll
                for (int e = 0; e < PL; ++e) asm volatile("" : "+v"(acc[e]));  // keep the update here
            };
            // A streamed batch: the next one's loads are issued before its row words are
            // awaited, so the exchange passes under them.  (A third buffer, with two
            // batches in flight, measured slower: 17.7 -> 22.2 us per iteration at 16 x
            // 1024 x 2048, 38.7 -> 44.0 at 4 x 4096 x 4096.)
            auto batch = [&](const float(&x)[KB][PL], int k0, float(&next)[KB][PL]) {
                const float own = dots(x);
                if (C > 1) rg.put(rowx, own, k0, nk, tag, local_row);
                load_rows(a.plan, k0 + KB, next);
                finish(x, k0, own);
            };
            float x[KB][PL], y[KB][PL];
            if (RR < nk) load_rows(a.plan, RR, x);
            // rows in registers, under the first streamed batch's loads: every batch is
            // published before the first is awaited
            if constexpr (RR > 0) {
                float own[RR / KB];
#pragma unroll
                for (int q = 0; q < RR / KB; ++q) {
                    own[q] = dots(xr[q]);
                    if (C > 1) rg.put(rowx, own[q], q * KB, nk, tag, local_row);
                }
#pragma unroll
                for (int q = 0; q < RR / KB; ++q) finish(xr[q], q * KB, own[q]);
            }
            for (int k = RR; k < nk; k += 2 * KB) {
                batch(x, k, y);
                if (k + KB < nk) batch(y, k + KB, x);
            }
            // a row factor out of range: the tile's column sums become NaN
            if (__any(bad)) {
#pragma unroll
                for (int e = 0; e < PL; ++e) acc[e] = __builtin_nanf("");
            }
        }
        if (__syncthreads_or(left)) {  // to the log domain, which does this iteration's rows again
            if (!leave)
                for (int j = threadIdx.x; j < nc; j += kThreads) lds_v[prev * seg + j] = logf(lds_v[prev * seg + j]);
            rows_to_u(t - 1);
            scal = leave = false;
            t0 = t;
            break;
        }
        // a row per thread (in the batches, each wave forms its rows' one after the
        // other: 144 x 400 x 450 629 -> 614 us per call, 4 x 1024 x 16384 5057 -> 4974)
        if (c == 0)
            for (int l = threadIdx.x; l < nrows; l += kThreads) {
                const float4 q = lds_row4[l];
                put_u(t, u_of(lds_la[l], q.y, cur ? q.w : q.z), l);
            }
        word_t dpre[res::kDeltaPrefetch];
        if (test && wave == 0) prefetch_deltas(t, dpre);
        const unsigned logs = columns(std::true_type{}, t);
        if (test && wave == 0) finish_deltas(t, dpre);
        dead = __any(dead);
        const bool flagged = __syncthreads_or(logs != 0);
        if (test && scratch[0] < a.tol) {  // the stop test of iteration t-1 fired
            used = t - 1;
            conv = 1;
            break;
        }
        if (flagged) {  // the rest of the tile's factors to v as well
            leave = true;
#pragma unroll
            for (int r = 0; r < kColsPerThread; ++r) {
                const int j = threadIdx.x + r * kThreads;
                if (j < nc && !((logs >> r) & 1u)) lds_v[cur * seg + j] = logf(lds_v[cur * seg + j]);
            }
        }
    }
    if (!scal) {
        __syncthreads();
        for (int t = t0; t <= a.max_iter; ++t) {
            const int cur = t & 1, prev = cur ^ 1;
            const unsigned tag = unsigned(t);
            const bool test = check && t >= 2;
            clear();
            // Log domain, as pst::forward's rows: y = (K + v) log2 e, a tile's maximum
            // and sum of a row in two words, folded over the tiles.
            word_t* rowl = a.rowl + size_t(cur) * a.B * a.M * C * 2;
            float v2[PL];
            Rw::load(lds_v + prev * seg, lane, nc, v2, 0.0f);
#pragma unroll
            for (int e = 0; e < PL; ++e) v2[e] *= kLog2E;
            // (the next batch's loads pass under this one's exchange: 16 x 1024 x 2048
            // 28.5 -> 26.2 us per iteration, 4 x 1024 x 16384 55 -> 51)
            auto batch = [&](float(&x)[KB][PL], int k0, float(&next)[KB][PL]) {
                load_rows(a.X, k0 + KB, next);
                mask_rows(x);
                float q[KB];
#pragma unroll
                for (int r = 0; r < KB; ++r) {
                    q[r] = -FLT_MAX;
#pragma unroll
                    for (int e = 0; e < PL; ++e) {
                        x[r][e] = fmaf(x[r][e], kscale2, v2[e]);
                        q[r] = fmaxf(q[r], x[r][e]);
                    }
                }
                const float m_own = res::transposed_reduce<KB>(q, OpMax{});
#pragma unroll
                for (int r = 0; r < KB; ++r) {
                    const float mr = read_lane(m_own, res::lane_of_slot<KB>(r));
                    q[r] = 0.0f;
#pragma unroll
                    for (int e = 0; e < PL; ++e) {
                        x[r][e] = __builtin_amdgcn_exp2f(x[r][e] - mr);
                        q[r] += x[r][e];
                    }
                }
                const float s_own = res::transposed_sum<KB>(q);
                float m, s_sum;
                if (C > 1) {
                    const bool on = rg.reads(k0, nk);
                    rg.put(rowl, m_own, k0, nk, tag, local_row, 2, 0);
                    rg.put(rowl, s_own, k0, nk, tag, local_row, 2, 1);
                    const float mt = rg.get(rowl, k0, nk, tag, a.spin_limit, a.status, dead, 2, 0);
                    const float st = rg.get(rowl, k0, nk, tag, a.spin_limit, a.status, dead, 2, 1);
                    m = group_reduce(on ? mt : -FLT_MAX, rg.lg, OpMax{});
                    s_sum = group_reduce(on ? st * __builtin_amdgcn_exp2f(mt - m) : 0.0f, rg.lg, OpSum{});
                } else {
                    m = rg.to_group(m_own);
                    s_sum = rg.to_group(s_own);
                }
                const bool ok = rg.group_ok(k0, nk);
                const int l = ok ? rg.group_row(k0) : 0;
                const float lga = lds_la[l];
                const float lg2 = __builtin_amdgcn_logf(fmaxf(s_sum, sk::kSumFloor));
                const float u = lga - kLn2 * (m + lg2);
                if (ok) {
                    dmax = fmaxf(dmax, fabsf(u - lds_u[prev * R + l]));
                    if (rg.leader()) {
                        lds_u[cur * R + l] = u;
                        if (c == 0) put_u(t, u, l);
                    }
                }
                const float w = ok ? __builtin_amdgcn_exp2f(fmaf(lga, kLog2E, -lg2)) : 0.0f;
#pragma unroll
                for (int r = 0; r < KB; ++r) {
                    const float mr = read_lane(m_own, res::lane_of_slot<KB>(r));
                    const float wr =
                        k0 + r < nk ? rg.of_group(w, r) * __builtin_amdgcn_exp2f(mr - rg.of_group(m, r)) : 0.0f;
#pragma unroll
                    for (int e = 0; e < PL; ++e) acc[e] = fmaf(x[r][e], wr, acc[e]);
                }
#pragma unroll
                for (int e = 0; e < PL; ++e) asm volatile("" : "+v"(acc[e]));  // keep the update here
            };
            float x[KB][PL], y[KB][PL];
            if (nk > 0) load_rows(a.X, 0, x);
            for (int k = 0; k < nk; k += 2 * KB) {
                batch(x, k, y);
                if (k + KB < nk) batch(y, k + KB, x);
            }
            word_t dpre[res::kDeltaPrefetch];
            if (test && wave == 0) prefetch_deltas(t, dpre);
            columns(std::false_type{}, t);
            if (test && wave == 0) finish_deltas(t, dpre);
            dead = __any(dead);
            __syncthreads();
            if (test && scratch[0] < a.tol) {
                used = t - 1;
                conv = 1;
                break;
            }
        }
        // (the rows kept in registers are E, which the log domain does not use: their
        // registers are free for its second buffer)
#pragma unroll
        for (int q = 0; q < RR / KB; ++q)
#pragma unroll
            for (int r = 0; r < KB; ++r)
#pragma unroll
                for (int e = 0; e < PL; ++e) xr[q][r][e] = 0.0f;
    }
    __syncthreads();
    if (leave) {
        rows_to_u(used);
        scal = false;
        __syncthreads();
    }
    if (check && conv == 0 && a.max_iter >= 1) {
        // the last iteration's deltas decide `converged`
        word_t* ds = a.dxchg + size_t(a.max_iter % res::kDeltaSlots) * G;
        if (wave == 0) {
            float m = 0.0f;
            for (int g = lane; g < G; g += kWave)
                m = res::OpMaxNan{}(m, res::collect(ds + g, unsigned(a.max_iter), a.spin_limit, a.status, dead));
            m = wave_reduce(m, res::OpMaxNan{});
            if (lane == 0) scratch[0] = m;
        }
        __syncthreads();
        conv = scratch[0] < a.tol ? 1 : 0;
    }

    // P = E w V, or safe_exp(K + u + v) (kernels.cu:755-775) in the log domain,
    // and this workgroup's share of sum(P C).
    const int par = used & 1;
    if (scal) {  // w of the plan's rows in the place of a
        for (int l = threadIdx.x; l < nrows; l += kThreads) {
            const float4 q = lds_row4[l];
            lds_row4[l].x = q.x / (par ? q.w : q.z);
        }
        __syncthreads();
    }
    const bool failed = __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    float vf[PL];
    Rw::load(lds_v + par * seg, lane, nc, vf, 0.0f);
    if (a.v_out && s == 0)
        for (int j = threadIdx.x; j < nc; j += kThreads) {
            const float vj = lds_v[par * seg + j];
            a.v_out[bN + c0 + j] = scal ? logf(vj) : vj;
        }
    if (a.u_out && c == 0)
        for (int l = threadIdx.x; l < nrows; l += kThreads) {
            const float4 q = lds_row4[l];
            a.u_out[bM + row0 + l] = scal ? u_of(lds_la[l], q.y, par ? q.w : q.z) : lds_u[par * R + l];
        }
    const float csign = a.scores_kind < 0 ? 1.0f : -1.0f;  // C = -log_alpha
    float cacc = 0.0f;
    // `e` holds the row's E, or (from_scores) its scores, whose E is formed again: the
    // cost reads them in any case, and E need not be read as well.
    auto write_row = [&](int l, float(&x)[PL], const float(&sc)[PL], bool from_scores, int ln) {
        const float4 q = lds_row4[l];
        const float wi = q.x, ui = scal ? 0.0f : lds_u[par * R + l];
        const auto row = kernel.row(q.y);
        float crow = 0.0f;  // (one chain over all of a lane's entries loses the small ones: -3.3e-7 of the cost)
#pragma unroll
        for (int e = 0; e < PL; ++e) {
            float p;
            if (scal) p = ((from_scores ? kernel.e(sc[e], row) : x[e]) * wi) * vf[e];
            else p = safe_exp((sc[e] * a.kscale + ui) + vf[e]);
            if (a.cost_partial && Rw::valid(ln, e, nc)) crow = fmaf(p, csign * sc[e], crow);
            x[e] = failed ? __builtin_nanf("") : p;
        }
        cacc += crow;
        Rw::store(a.plan + tile0 + size_t(l) * a.N, ln, nc, x);
    };
    const bool scores = a.cost_partial || !scal;
#pragma unroll
    for (int q = 0; q < RR / KB; ++q) {
        float sc[KB][PL];
        if (scores && nk > 0) load_rows(a.X, q * KB, sc);
#pragma unroll
        for (int r = 0; r < KB; ++r)
            if (q * KB + r < nk) write_row(wave + kWaves * (q * KB + r), xr[q][r], sc[r], false, pst::opaque_lane());
    }
    for (int k = RR; k < nk; k += KB) {
        float x[KB][PL];
        load_rows(scores ? a.X : a.plan, k, x);
#pragma unroll
        for (int r = 0; r < KB; ++r)
            if (k + r < nk) write_row(wave + kWaves * (k + r), x[r], x[r], scores, pst::opaque_lane());
    }
    if (scal) {
        // An entry whose E was flushed to 0 may be a float's itself where w V passes 1:
        // formed from its score, in a pass of its own over such rows (inside the one
        // above, its branch cost every call 5 of 147 us at 16 x 1024 x 2048).
        float vmax = vf[0];
#pragma unroll
        for (int e = 1; e < PL; ++e) vmax = fmaxf(vmax, vf[e]);
        vmax = wave_max(vmax);
        bool any = false;
        for (int k = lane; k < nk; k += kWave) any = any || lds_row4[wave + kWaves * k].x * vmax > 1.0f;
        for (int k = 0; __any(any) && k < nk; ++k) {
            const int l = wave + kWaves * k;
            const float4 q = lds_row4[l];
            if (!(q.x * vmax > 1.0f)) continue;
            const size_t at = tile0 + size_t(l) * a.N;
            float p[PL], sc[PL];
            load_row(a.plan + at, p);
            load_row(a.X + at, sc);
            const float u = u_of(lds_la[l], q.y, par ? q.w : q.z);
#pragma unroll
            for (int e = 0; e < PL; ++e)
                if (p[e] == 0.0f && q.x * vf[e] > 1.0f) p[e] = safe_exp((sc[e] * a.kscale + u) + logf(vf[e]));
            Rw::store(a.plan + at, lane, nc, p);
        }
    }
    if (a.cost_partial) {
        const float cs = block_reduce<kWaves>(wave_sum(cacc), scratch + 16, OpSum{});
        if (threadIdx.x == 0) a.cost_partial[gid] = failed ? __builtin_nanf("") : cs;
    }
    if (gid == 0 && threadIdx.x == 0) {
        *a.iters_used = failed ? -1 : used;  // -1: an exchange timed out, the outputs are NaN
        *a.converged = conv;
    }
}

}  // namespace til
}  // namespace dot_amd
