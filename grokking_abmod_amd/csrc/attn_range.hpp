// Which (sequence, head) pairs of a long prefill run on split FP16 operands
// (attn_split.hip) and which on FP32 ones (attn_mfma.hip): both kernels are
// launched and each leaves the other's pairs alone.
#pragma once

#include <hip/hip_runtime.h>

namespace meshgpt::kern {

constexpr int kSplitKeys = 64;     // keys of a tile
constexpr int kSplitSpread = 10;   // see attn_split.hip
constexpr int kSplitTiny = 4;      // see attn_split.hip
constexpr int kBadRange = 4096;    // a tile whose values need the FP32 kernel
constexpr int kNoRow = 2048;       // a tile of zeros

// The exponent E of the largest |v| of a pair (v < 2^E) from its tiles' ranges
// (x: the tile's largest, y: its smallest row's largest), the same in every
// lane; false where the pair takes the FP32 kernel.
__device__ __forceinline__ bool pair_splits(const int2 *tile_range, int tiles, int lane, int &E) {
    int top = -kNoRow, low = kNoRow;
    for (int t = lane; t < tiles; t += 64) {
        const int2 r = tile_range[t];
        top = max(top, r.x);
        low = min(low, r.y);
    }
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
        top = max(top, __shfl_xor(top, k, 64));
        low = min(low, __shfl_xor(low, k, 64));
    }
    E = __builtin_amdgcn_readfirstlane(top);
    return E != kBadRange && E - __builtin_amdgcn_readfirstlane(low) <= kSplitSpread;
}

}  // namespace meshgpt::kern
