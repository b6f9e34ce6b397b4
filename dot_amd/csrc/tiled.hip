// Launch of the tiled persistent kernels (a translation unit of their own).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "coop.hpp"
#include "host.hpp"
#include "tiled.cuh"
#include "tiled.hpp"

namespace dot_amd {
namespace {

constexpr int kLdsBytes = 160 * 1024;
constexpr int kMinStripRows = res::kWaves;  // a row for every wave

struct Words {
    size_t rowx, rowl, part, res, uslot, dxchg, xcc, status, cost, total;
};

Words words_of(const TiledCfg& c, int B, int M, int N) {
    const size_t G = size_t(B) * c.ST * c.C, rows = size_t(B) * M;
    Words w{};
    w.rowx = 0;
    w.rowl = w.rowx + (c.C > 1 ? 2 * rows * c.C : 0);
    w.part = w.rowl + (c.C > 1 ? 4 * rows * c.C : 0);
    w.res = w.part + 2 * G * c.seg;
    w.uslot = w.res + 2 * size_t(B) * N;
    w.dxchg = w.uslot + 2 * rows;
    w.xcc = w.dxchg + res::kDeltaSlots * G;
    w.status = w.xcc + G;
    w.cost = w.status + 1;  // [G] floats, not cleared
    w.total = w.cost + (G + 1) / 2;
    return w;
}

}  // namespace

// Tiles of at most 512 columns (8 floats per lane) while sixteen of them make a
// row, of at most 1024 beyond: a batch of a wave is four rows of a narrow tile
// or two of a wide one, and the narrow one amortises a batch's fixed work over
// as many elements with half the accumulator (per iteration, narrow against
// wide: 16 x 1024 x 2048 17.7 and 20.6 us, 4 x 4096 x 4096 38.7 and 41.5 us).
// As many strips as the CUs hold, each with at least a row per wave.
TiledCfg tiled_config(int B, int M, int N) {
    TiledCfg c;
    const char* env = std::getenv("DOT_AMD_TILED");
    if (env && env[0] == '0') return c;
    if (B < 1 || M < 1 || N < 4) return c;
    // a strip's tiles share an XCD (til::forward), so strips are counted per XCD
    const int xcd_cus = device_cus() / res::kXcds;
    if (xcd_cus <= 0) return c;
    c.narrow = N <= 512 || (N > 1024 && N <= 512 * til::kMaxTiles);
    const int width = c.narrow ? 512 : 1024;
    c.C = (N + width - 1) / width;
    if (c.C > til::kMaxTiles) return c;
    const int all = xcd_cus / c.C * res::kXcds;
    if (B > all) return c;
    c.seg = ((N + c.C - 1) / c.C + 3) & ~3;
    const int strips = std::min({all / B, til::kMaxStrips, std::max(M / kMinStripRows, 1)});
    // byte offsets of the row words are 32-bit
    if (size_t(B) * M * c.C * 2 * sizeof(unsigned long long) > (size_t(1) << 31)) return c;
    c.R = (M + strips - 1) / strips;
    c.ST = (M + c.R - 1) / c.R;
    c.ok = true;
    return c;
}

size_t tiled_forward_bytes(const TiledCfg& c, int B, int M, int N) {
    return words_of(c, B, M, N).total * sizeof(unsigned long long);
}

bool launch_tiled_forward(til::FwdArgs& a, const TiledCfg& c, bool vec4, bool cost, void* words,
                          float** cost_partial, hipStream_t stream) {
    const int G = a.B * c.ST * c.C;
    const int grid = (a.B * c.ST + res::kXcds - 1) / res::kXcds * res::kXcds * c.C;
    const Words w = words_of(c, a.B, a.M, a.N);
    auto* base = static_cast<unsigned long long*>(words);
    a.rowx = base + w.rowx;
    a.rowl = base + w.rowl;
    a.part = base + w.part;
    a.res = base + w.res;
    a.uslot = base + w.uslot;
    a.dxchg = base + w.dxchg;
    a.xcc = base + w.xcc;
    a.status = reinterpret_cast<int*>(base + w.status);
    a.cost_partial = cost ? reinterpret_cast<float*>(base + w.cost) : nullptr;
    *cost_partial = a.cost_partial;
    a.G = G;
    a.C = c.C;
    a.ST = c.ST;
    a.R = c.R;
    a.seg = c.seg;
    const size_t lds = til::fwd_lds_floats(c.seg, c.ST, c.R) * sizeof(float);
    if (lds > size_t(kLdsBytes)) return false;
    bool ok = false;
    auto launch = [&](auto kernel) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, res::kThreads, lds) != hipSuccess ||
            per_cu < 1 || int64_t(per_cu) * device_cus() < grid)
            return;
        fill_zero_words(words, 2 * w.cost, stream);
        ProfScope prof("sk_fwd_tiled", stream);
        ok = launch_persistent(kernel, a, grid, res::kThreads, lds, stream);
    };
    // Batches of KB rows and RR rows kept in registers, us per iteration (RR = RR / 2,
    // 0, 1.5 RR; then KB / 2, 2 KB at the same RR): 16 x 1024 x 2048 17.6 (19.3, 21.1,
    // 24.8; 23.0, 52.7), 4 x 4096 x 4096 39.5 (41.4, 42.2, 47.8; 50.7, 78), 4 x 1024 x
    // 16384 39.6 (40.9, 43.4, 55; 47.0, 79).  Scalar rows: KB / 2 and 2 KB are slower as
    // well; RR = 8 and 4 are faster at rows of 2047 (18.1 for 19.7) and 16381 (40.7 for
    // 44.4) and equal at 450 and 1001.
    if (vec4) {
        if (c.narrow) launch(til::forward<4, 2, 4, 8>);
        else launch(til::forward<4, 4, 2, 4>);
    } else {
        if (c.narrow) launch(til::forward<1, 8, 4, 4>);
        else launch(til::forward<1, 16, 2, 0>);
    }
    return ok;
}

}  // namespace dot_amd
