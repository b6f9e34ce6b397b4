// Host side of the tiled persistent forward (tiled.cuh): shapes it takes, its
// exchange words and its launch.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace dot_amd {

struct TiledCfg {
    bool ok = false;
    int C = 1, ST = 1, R = 1, seg = 1;  // tiles per row, strips, rows per strip, columns per tile
    bool narrow = false;                // tiles of at most 512 columns (8 floats per lane)
};

TiledCfg tiled_config(int B, int M, int N);

// Bytes of the exchange words of a launch of this configuration.
size_t tiled_forward_bytes(const TiledCfg& c, int B, int M, int N);

namespace til {
struct FwdArgs;
}

// Launches the forward on `words` (tiled_forward_bytes; cleared here); `a` has
// everything but the tile shape and the words.  With `cost`, *cost_partial is
// set to the [B, ST C] partial sums of P C that the launch writes.  False when
// the device cannot hold the grid (nothing is launched).
bool launch_tiled_forward(til::FwdArgs& a, const TiledCfg& c, bool vec4, bool cost, void* words,
                          float** cost_partial, hipStream_t stream);

}  // namespace dot_amd
