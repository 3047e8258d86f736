// The operand order of the product with several vectors (internal; the public ABI is include/).
//
// Vectors [batch, cols] fp16 as v_mfma_f32_16x16x32_f16 takes them: per 64 columns and 16 vectors one block
// of 128 pieces of 16 bytes, piece s * 64 + 16 q + n = columns 16 q + 8 s .. + 7 of vector n, blocks of the
// same columns next to each other.  A wave's two operand loads per block are then 1 KB of consecutive
// memory each.  Columns and vectors that do not exist are zero.
#pragma once

#include "macko_common.h"

namespace macko {

constexpr int kBlockPieces = 128;
__host__ __device__ inline int packed_tiles(int batch) { return (batch + 15) / 16; }
__host__ __device__ inline int packed_steps(int cols) { return (cols + 63) / 64; }
inline size_t packed_bytes(int cols, int batch) { return (size_t)packed_tiles(batch) * (size_t)packed_steps(cols) * (kBlockPieces * 16); }

// piece (8 columns) p of vector n
__device__ __forceinline__ size_t packed_piece(int p, int n, int tiles)
{
    return ((size_t)(p >> 3) * (size_t)tiles + (size_t)(n >> 4)) * kBlockPieces + (size_t)((p & 1) * 64 + ((p >> 1) & 3) * 16 + (n & 15));
}

// The gate of a Llama layer.
__device__ __forceinline__ float silu_mul(float gate, float up) { return gate / (1.0f + __expf(-gate)) * up; }

// The halves of a 16-byte piece from element `by` on, zeros behind them (by >= 8: all zero).
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int by)
{
    unsigned long long lo = v.x | ((unsigned long long)v.y << 32), hi = v.z | ((unsigned long long)v.w << 32);
    if (by >= 4) {
        lo = hi;
        hi = 0;
        by -= 4;
    }
    if (by >= 4) lo = 0, by = 0;
    if (by > 0) {
        const int s = 16 * by;
        lo = (lo >> s) | (hi << (64 - s));
        hi >>= s;
    }
    return u32x4{(u32)lo, (u32)(lo >> 32), (u32)hi, (u32)(hi >> 32)};
}

}  // namespace macko
